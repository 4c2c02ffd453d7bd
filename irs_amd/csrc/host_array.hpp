// A host array for results that a device copy fills: contents undefined until
// then, large ones on huge pages. A std::vector writes zeros first and takes a
// page fault per 4 KB (a 400 MB map: 94 ms until it was on the host, most of it
// that; 24 MB of FP64 maps: 5.3 ms).
#pragma once

#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <new>
#include <utility>

namespace mlens
{

template <typename T>
class HostArray
{
public:
	HostArray() = default;
	~HostArray() { clear(); }
	HostArray(const HostArray&) = delete;
	HostArray& operator=(const HostArray&) = delete;

	// n elements with undefined contents
	void resize(size_t n)
	{
		if (n == size_) return;
		clear();
		if (n == 0) return;
		constexpr size_t HUGE = size_t(2) << 20;
		const size_t bytes = n * sizeof(T);
		if (bytes >= 2 * HUGE)
		{
			const size_t rounded = (bytes + HUGE - 1) / HUGE * HUGE;
			ptr_ = static_cast<T*>(std::aligned_alloc(HUGE, rounded));
			if (ptr_) (void)madvise(ptr_, rounded, MADV_HUGEPAGE);   // advice: small pages do as well
		}
		else
			ptr_ = static_cast<T*>(std::malloc(bytes));
		if (!ptr_) throw std::bad_alloc();
		size_ = n;
	}
	// n elements that fill(data) writes; zeros if it throws
	template <typename F>
	void fill(size_t n, F fill)
	{
		resize(n);
		try
		{
			fill(ptr_);
		}
		catch (...)
		{
			if (ptr_) std::memset(static_cast<void*>(ptr_), 0, n * sizeof(T));
			throw;
		}
	}
	void clear()
	{
		std::free(ptr_);
		ptr_ = nullptr;
		size_ = 0;
	}
	bool empty() const { return size_ == 0; }
	size_t size() const { return size_; }
	T* data() { return ptr_; }
	const T* data() const { return ptr_; }
	T& operator[](size_t i) { return ptr_[i]; }

private:
	T* ptr_ = nullptr;
	size_t size_ = 0;
};

}  // namespace mlens
