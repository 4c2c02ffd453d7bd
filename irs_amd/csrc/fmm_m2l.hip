// M2L as batched GEMMs on the matrix cores (fmm.cuh:281-374 restated as
// matrix products).
//
// A source f in the M2L list of a target t sits at the target's level, at
// dz = (c_f - c_t) / h = 2 (a + i b) with integers |a|, |b| <= 3 and
// max(|a|, |b|) >= 2: 40 offsets. In node-normalised units the translation
// is linear in the source multipole b and depends only on the offset:
//
//   c_0 += sum_{k>=1} b_k (-dz)^-k + b_0 log(-dz) + b_0 log h
//   c_l += sum_{k>=1} C(l+k-1, k-1) b_k (-dz)^-k dz^-l - b_0 / (l dz^l),  l >= 1
//
// so c += M_o b with 40 fixed (p+1) x (p+1) complex matrices M_o, plus the
// level-dependent b_0 log h term. Complex products run as real products of
// the stacked form [Mr -Mi; Mi Mr] [b_re; b_im], padded to a multiple of 16.
//
// Sources sit at their target's level and the matrices do not depend on it, so
// one launch translates every level. A block takes 16 (or 32) sibling groups
// (the four children of a node, consecutive) and one of the four quadrants:
// targets of the same quadrant share the 27 offsets their M2L lists can hold,
// where a mixed block would step through all 40. Wave w owns row tile w of the
// block's targets (the columns of a 16 x 16 output tile): for each offset that
// some target has, it accumulates M_o b in registers, offsets ascending, so no
// target row is written by two waves and no atomics are needed. The block
// gathers each offset's sources into LDS once for all its waves (two buffers,
// one barrier an offset), each wave its rows of the matrix into registers, both
// an offset ahead. The offset matrices (1.3 MB) stay in L2. 1.28e6 stars at
// p = 30 (2.2e7 pairs): 5.1 ms, 43% of the FP64 MFMA time of the padded
// products; 13.0 ms with one launch per level, mixed quadrants and every wave
// computing all row tiles of its own targets, 10 ms with the sources gathered
// by each wave. 7e3 stars at p = 20, where the chain of offsets is the time:
// 54 us against six launches of 265 us.
// The MFMA shape is 16 x 16 x 4 in FP32 (v_mfma_f32_16x16x4_f32) or FP64
// (v_mfma_f64_16x16x4_f64); both take A[i][k] from lane i + 16 k and B[k][j]
// from lane j + 16 k. Lane l gets back D[4 (l / 16) + r][l % 16] in FP32 and
// D[(l / 16) + 4 r][l % 16] in FP64, r = 0..3 (checked on the device).
#include "engine.hpp"
#include "device_math.hpp"

#include <complex>
#include <vector>

namespace mlens
{

namespace
{

constexpr int M2L_OFFSETS = 40;
constexpr int M2L_LIST = 27;   // longest M2L list (tree_node.cuh:41-49)

inline int m2l_kp(int p) { return (2 * (p + 1) + 15) / 16 * 16; }

// offset (a, b), |a|, |b| <= 3, to its index 0..39, or -1 for the 3 x 3 near block
__host__ __device__ inline int m2l_offset_index(int a, int b)
{
	if (a < -3 || a > 3 || b < -3 || b > 3) return -1;
	if (a >= -1 && a <= 1 && b >= -1 && b <= 1) return -1;
	int idx = (b + 3) * 7 + (a + 3);   // 0..48 over the 7 x 7 block
	// drop the 9 near entries that precede idx
	int before = 0;
	for (int bb = -1; bb <= 1; bb++)
		for (int aa = -1; aa <= 1; aa++)
			if ((bb + 3) * 7 + (aa + 3) < idx) before++;
	return idx - before;
}

template <typename T>
struct MfmaVec;
template <>
struct MfmaVec<float>
{
	typedef float v4 __attribute__((ext_vector_type(4)));
	static __device__ __forceinline__ v4 mfma(float a, float b, v4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
	static __device__ __forceinline__ int row(int kq, int r) { return kq * 4 + r; }
};
template <>
struct MfmaVec<double>
{
	typedef double v4 __attribute__((ext_vector_type(4)));
	static __device__ __forceinline__ v4 mfma(double a, double b, v4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
	static __device__ __forceinline__ int row(int kq, int r) { return kq + 4 * r; }
};

/*
out[node][2 row + c] = row `row` (real c = 0, imaginary 1) of the M2L sum of nodes
first + 4 g + q, g < groups. KP: stacked size (2 (p + 1) rounded up to 16), KP / 16
waves per block; NT: column tiles (16 targets each) per block. The four quadrants of
the same groups, which share most of their sources, are consecutive pieces of work, and
each XCD (blocks go to the eight in turn) takes a contiguous run of them, so that its
L2 holds the multipoles that they read over and over.
count[0] collects the list entries, the low bit of count[1] a source that is not at
one of the 40 offsets.
*/
template <typename T, int KP, int NT>
__global__ __launch_bounds__(KP * 4) void k_m2l(const T* __restrict__ At, const double* __restrict__ mult, double* __restrict__ out,
	const double* __restrict__ cx, const double* __restrict__ cy, const double* __restrict__ hl, const int* __restrict__ nm2l,
	const int* __restrict__ m2l, int first, int groups, int p, unsigned long long* __restrict__ count)
{
	using V = typename MfmaVec<T>::v4;
	constexpr int KS = KP / 4, TARGETS = 16 * NT, THREADS = KP * 4, STAGE = TARGETS * KP / THREADS;
	// 2 modulo 32 eight-byte banks: the 16 targets and two rows a half-wave reads fall on 32 of them
	constexpr int STRIDE = (KP + 31) / 32 * 32 + 2;
	__shared__ T gathered[2][TARGETS * STRIDE];
	__shared__ int src[M2L_OFFSETS][TARGETS];   // the source of each target at each offset, or -1
	__shared__ unsigned active[2];              // offsets that some target has
	__shared__ unsigned found;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int col = lane & 15, kq = lane >> 4;
	const int run = int(gridDim.x) / 8;   // pieces per XCD (the grid is a multiple of 8)
	const int piece = int(blockIdx.x % 8) * run + int(blockIdx.x / 8);
	const int g0 = (piece >> 2) * TARGETS, q = piece & 3;
	if (g0 >= groups) return;
	for (int i = threadIdx.x; i < M2L_OFFSETS * TARGETS; i += blockDim.x) src[i / TARGETS][i % TARGETS] = -1;
	for (int i = threadIdx.x; i < 2 * TARGETS * STRIDE; i += blockDim.x) gathered[0][i] = T(0);
	if (threadIdx.x == 0) active[0] = active[1] = found = 0;
	__syncthreads();
	for (int i = threadIdx.x; i < M2L_LIST * TARGETS; i += blockDim.x)
	{
		const int c = i / M2L_LIST, j = i - c * M2L_LIST;
		if (g0 + c >= groups) continue;
		const int t = first + 4 * (g0 + c) + q;
		if (j >= nm2l[t]) continue;
		const int f = m2l[M2L_LIST * (long long)t + j];
		const double h2 = 2 * hl[t];
		const int o = m2l_offset_index(int(lrint((cx[f] - cx[t]) / h2)), int(lrint((cy[f] - cy[t]) / h2)));
		atomicAdd(&found, 1u);
		if (o < 0 || hl[f] != hl[t])
		{
			atomicOr(reinterpret_cast<unsigned*>(count + 1), 1u);
			continue;
		}
		src[o][c] = f;
		atomicOr(&active[o >> 5], 1u << (o & 31));
	}
	__syncthreads();
	if (threadIdx.x == 0 && found) atomicAdd(count, (unsigned long long)found);
	unsigned long long todo = ((unsigned long long)__builtin_amdgcn_readfirstlane(active[1]) << 32) |
		(unsigned)__builtin_amdgcn_readfirstlane(active[0]);
	const int P = p + 1;
	V acc[NT];
	double sum0[NT];   // sum of the sources' b_0, for the b_0 log h term (its lanes: row 0)
#pragma unroll
	for (int n = 0; n < NT; n++)
	{
		acc[n] = V{0, 0, 0, 0};
		sum0[n] = 0;
	}
	// the operands of one offset: this wave's rows of the matrix, and this thread's
	// share of the sources' multipoles
	struct Operands
	{
		T a[KS];
		T b[STAGE];
		double b0[NT];
	};
	auto load = [&](int o, Operands& x) {
		const T* Ao = At + ((long long)o * KP + kq) * KP + wave * 16 + col;
#pragma unroll
		for (int ks = 0; ks < KS; ks++) x.a[ks] = Ao[(long long)ks * 4 * KP];
#pragma unroll
		for (int r = 0; r < STAGE; r++)
		{
			const int e = threadIdx.x + r * THREADS, c = e / KP, j = e % KP;
			const int s = src[o][c];
			x.b[r] = (s >= 0 && j < 2 * P) ? T(mult[(long long)s * P * 2 + j]) : T(0);
		}
#pragma unroll
		for (int n = 0; n < NT; n++)
		{
			const int s = wave == 0 ? src[o][n * 16 + col] : -1;
			x.b0[n] = s >= 0 ? mult[(long long)s * P * 2] : 0.0;
		}
	};
	// row k < P of a stacked multipole is Re b_k, then Im b_(k - P); rows past 2 P stay zero
	auto stage = [&](const Operands& x, T* to) {
#pragma unroll
		for (int r = 0; r < STAGE; r++)
		{
			const int e = threadIdx.x + r * THREADS, c = e / KP, j = e % KP;
			if (j < 2 * P) to[c * STRIDE + ((j & 1) ? P + (j >> 1) : (j >> 1))] = x.b[r];
		}
	};
	auto multiply = [&](const Operands& x, const T* from) {
#pragma unroll
		for (int ks = 0; ks < KS; ks++)
#pragma unroll
			for (int n = 0; n < NT; n++)
				acc[n] = MfmaVec<T>::mfma(x.a[ks], from[(n * 16 + col) * STRIDE + ks * 4 + kq], acc[n]);
#pragma unroll
		for (int n = 0; n < NT; n++) sum0[n] += x.b0[n];
	};
	auto next = [&]() {
		const int o = __builtin_ctzll(todo);
		todo &= todo - 1;
		return o;
	};
	Operands x, y;
	bool have = todo != 0;
	if (have) load(next(), x);
	while (have)
	{
		// each buffer is written two barriers after its last readers passed one
		stage(x, gathered[0]);
		__syncthreads();
		bool more = todo != 0;
		if (more) load(next(), y);
		multiply(x, gathered[0]);
		if (!more) break;
		stage(y, gathered[1]);
		__syncthreads();
		have = todo != 0;
		if (have) load(next(), x);
		multiply(y, gathered[1]);
	}
#pragma unroll
	for (int n = 0; n < NT; n++)
	{
		const int g = g0 + n * 16 + col;
		if (g >= groups) continue;
		const int t = first + 4 * g + q;
		double* c = out + (long long)t * P * 2;
		// the b_0 log h term in FP64 from the FP64 multipoles (b_0 is real), added after the product
		double extra;
		{
#pragma clang fp contract(off)
			extra = sum0[n] * log(hl[t]);
		}
#pragma unroll
		for (int r = 0; r < 4; r++)
		{
			const int row = wave * 16 + MfmaVec<T>::row(kq, r);
			const double v = double(acc[n][r]) + (row == 0 ? extra : 0.0);
			if (row < P)
				c[2 * row] = v;
			else if (row < 2 * P)
				c[2 * (row - P) + 1] = v;
		}
	}
}

// launches the instantiation for kp; wide: two column tiles per block
template <typename T>
void launch_m2l(int kp, bool wide, hipStream_t st, const T* At, const double* mult, double* out, const double* cx,
	const double* cy, const double* hl, const int* nm2l, const int* m2l, int first, int groups, int p, unsigned long long* count)
{
	auto go = [&](auto kernel, int targets) {
		kernel<<<unsigned((4 * ((groups + targets - 1) / targets) + 7) / 8 * 8), kp * 4, 0, st>>>(At, mult, out, cx, cy, hl, nm2l, m2l, first,
			groups, p, count);
	};
	switch (kp)
	{
	case 16: wide ? go(k_m2l<T, 16, 2>, 32) : go(k_m2l<T, 16, 1>, 16); break;
	case 32: wide ? go(k_m2l<T, 32, 2>, 32) : go(k_m2l<T, 32, 1>, 16); break;
	case 48: wide ? go(k_m2l<T, 48, 2>, 32) : go(k_m2l<T, 48, 1>, 16); break;
	default: wide ? go(k_m2l<T, 64, 2>, 32) : go(k_m2l<T, 64, 1>, 16); break;
	}
}

}  // namespace

namespace
{

// per offset: log(-dz), then (-dz)^-k and dz^-k, k < P
constexpr int M2L_POWERS = 1 + 2 * (MAX_EXPANSION_ORDER + 1);

/* The 40 offset matrices for order p (blockIdx.x = offset), stacked [Mr -Mi; Mi Mr], stored transposed At[col][row]
   and zero-padded to kp. The host sends the powers of the offsets (42 KB) and the binomials; building the matrices
   there and copying them took 0.4 ms of a small field's build. Contraction is off: the entries are those that the
   host's complex products give. */
template <typename T>
__global__ void k_m2l_matrices(const double* __restrict__ powers, const double* __restrict__ B, int p, int kp, T* __restrict__ A)
{
#pragma clang fp contract(off)
	const int o = blockIdx.x, P = p + 1;
	const double* w = powers + o * M2L_POWERS * 2;
	const double *ip = w + 2, *dzi = ip + 2 * P;
	T* Ao = A + (long long)o * kp * kp;
	for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < kp * kp; i += gridDim.y * blockDim.x)
	{
		const int col = i / kp, row = i - col * kp;
		double v = 0;
		if (col < 2 * P && row < 2 * P)
		{
			const int k = col % P, l = row % P;
			double re, im;
			if (l == 0)
			{
				re = k == 0 ? w[0] : ip[2 * k];
				im = k == 0 ? w[1] : ip[2 * k + 1];
			}
			else if (k == 0)
			{
				re = -dzi[2 * l] / double(l);
				im = -dzi[2 * l + 1] / double(l);
			}
			else
			{
				const int n = l + k - 1;
				const double c = B[n * (n + 1) / 2 + k - 1];
				const double a = c * ip[2 * k], b = c * ip[2 * k + 1], d = dzi[2 * l], e = dzi[2 * l + 1];
				re = a * d - b * e;
				im = a * e + b * d;
			}
			v = (col < P) == (row < P) ? re : (col < P ? im : -im);
		}
		Ao[i] = T(v);
	}
}

}  // namespace

void Engine::m2l_prepare(int p, bool f32)
{
	if (m2l_ready_p_ == p && m2l_ready_f32_ == f32) return;
	const int P = p + 1, kp = m2l_kp(p);
	std::vector<double>& w = m2l_host_;   // outlives the copy
	w.assign(size_t(M2L_OFFSETS) * M2L_POWERS * 2, 0.0);
	for (int b = -3; b <= 3; b++)
		for (int a = -3; a <= 3; a++)
		{
			const int o = m2l_offset_index(a, b);
			if (o < 0) continue;
			const std::complex<double> dz(2.0 * a, 2.0 * b), mdz = -dz, imdz = 1.0 / mdz;
			double* q = w.data() + size_t(o) * M2L_POWERS * 2;
			auto put = [&](int at, std::complex<double> v) {
				q[2 * at] = v.real();
				q[2 * at + 1] = v.imag();
			};
			put(0, std::log(mdz));
			std::complex<double> ipow = 1.0, dzinv = 1.0;
			for (int k = 0; k < P; k++)
			{
				put(1 + k, ipow);
				put(1 + P + k, dzinv);
				ipow = ipow * imdz;
				dzinv = dzinv / dz;
			}
		}
	m2l_powers_.alloc(w.size());
	MLENS_HIP_CHECK(hipMemcpyAsync(m2l_powers_.ptr, w.data(), w.size() * sizeof(double), hipMemcpyHostToDevice, stream_));
	const size_t n = size_t(M2L_OFFSETS) * kp * kp;
	const dim3 grid(M2L_OFFSETS, 4);
	if (f32)
	{
		m2l_af_.alloc(n);
		k_m2l_matrices<float><<<grid, 256, 0, stream_>>>(m2l_powers_.ptr, binom_.ptr, p, kp, m2l_af_.ptr);
	}
	else
	{
		m2l_ad_.alloc(n);
		k_m2l_matrices<double><<<grid, 256, 0, stream_>>>(m2l_powers_.ptr, binom_.ptr, p, kp, m2l_ad_.ptr);
	}
	MLENS_HIP_CHECK(hipGetLastError());
	m2l_ready_p_ = p;
	m2l_ready_f32_ = f32;
}

// the M2L sums of every node at level 2 and below, into local_ (k_local adds the rest)
void Engine::m2l_all(int p, bool f32)
{
	const int first = level_start_[2], groups = (num_nodes_ - first) / 4;
	if (groups <= 0) return;
	// two column tiles halve the matrix traffic once one tile per block fills the device
	const bool wide = groups >= 16 * num_cus_;
	if (f32)
		launch_m2l<float>(m2l_kp(p), wide, stream_, m2l_af_.ptr, mult_.ptr, local_.ptr, ncx_.ptr, ncy_.ptr, nhl_.ptr, nnm2l_.ptr,
			nm2l_.ptr, first, groups, p, m2l_count_.ptr);
	else
		launch_m2l<double>(m2l_kp(p), wide, stream_, m2l_ad_.ptr, mult_.ptr, local_.ptr, ncx_.ptr, ncy_.ptr, nhl_.ptr, nnm2l_.ptr,
			nm2l_.ptr, first, groups, p, m2l_count_.ptr);
	MLENS_HIP_CHECK(hipGetLastError());
}

}  // namespace mlens
