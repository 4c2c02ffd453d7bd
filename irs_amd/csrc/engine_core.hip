// Engine: device buffers, star field, quadtree build, FMM and leaf tables.
#include "engine.hpp"
#include "device_math.hpp"
#include "mass_functions.hpp"
#include "philox.hpp"

#include <algorithm>
#include <cstring>

namespace mlens
{

using dev::dcx;

template <typename T>
void DeviceBuffer<T>::alloc(size_t n)
{
	if (n <= count && ptr) return;
	free();
	if (n == 0) return;
	MLENS_HIP_CHECK(hipMalloc(&ptr, n * sizeof(T)));
	count = n;
}

template <typename T>
void DeviceBuffer<T>::free()
{
	if (ptr) (void)hipFree(ptr);
	ptr = nullptr;
	count = 0;
}

template struct DeviceBuffer<double>;
template struct DeviceBuffer<float>;
template struct DeviceBuffer<int>;
template struct DeviceBuffer<char>;
template struct DeviceBuffer<long long>;
template struct DeviceBuffer<unsigned long long>;
template struct DeviceBuffer<unsigned short>;

static inline unsigned blocks_for(long long n, int threads) { return unsigned((n + threads - 1) / threads); }

Engine::Engine()
{
	MLENS_HIP_CHECK(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
	MLENS_HIP_CHECK(hipEventCreate(&ev0_));
	MLENS_HIP_CHECK(hipEventCreate(&ev1_));
	int dev = 0;
	MLENS_HIP_CHECK(hipGetDevice(&dev));
	dev_ = dev;
	MLENS_HIP_CHECK(hipDeviceGetAttribute(&num_cus_, hipDeviceAttributeMultiprocessorCount, dev));
}

Engine::~Engine()
{
	if (stream_) (void)hipStreamSynchronize(stream_);
	if (ev0_) (void)hipEventDestroy(ev0_);
	if (ev1_) (void)hipEventDestroy(ev1_);
	if (m2l_ev0_) (void)hipEventDestroy(m2l_ev0_);
	if (m2l_ev1_) (void)hipEventDestroy(m2l_ev1_);
	if (stream_) (void)hipStreamDestroy(stream_);
}

/* ---------------------------------------------------------------------------
Stars
--------------------------------------------------------------------------- */
void Engine::upload_stars(const double* aos, int n)
{
	nstars_ = n;
	sx_.alloc(n);
	sy_.alloc(n);
	sm_.alloc(n);
	std::vector<double> a(n), b(n), c(n);
	for (int i = 0; i < n; i++)
	{
		a[i] = aos[3 * i];
		b[i] = aos[3 * i + 1];
		c[i] = aos[3 * i + 2];
	}
	MLENS_HIP_CHECK(hipMemcpy(sx_.ptr, a.data(), n * sizeof(double), hipMemcpyHostToDevice));
	MLENS_HIP_CHECK(hipMemcpy(sy_.ptr, b.data(), n * sizeof(double), hipMemcpyHostToDevice));
	MLENS_HIP_CHECK(hipMemcpy(sm_.ptr, c.data(), n * sizeof(double), hipMemcpyHostToDevice));
}

// star.cuh:64-107 with the Philox stream of philox.hpp
__global__ void k_generate_stars(double* sx, double* sy, double* sm, int n, int rectangular, double c_re, double c_im,
	int mf, double ml, double mu, double ms, uint32_t seed)
{
	int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	double u[4];
	star_uniforms(seed, i, u);
	double x1, x2;
	if (rectangular)
	{
		x1 = u[0] * 2 * c_re - c_re;
		x2 = u[1] * 2 * c_im - c_im;
	}
	else
	{
		double a = u[0] * 2 * PI;
		double r = sqrt(u[1]) * hypot(c_re, c_im);
		x1 = r * cos(a);
		x2 = r * sin(a);
	}
	sx[i] = x1;
	sy[i] = x2;
	sm[i] = sample_mass<double>(mf, u[2], ml, mu, ms);
}

void Engine::generate_stars(int n, int rectangular, double c_re, double c_im, int mf, double ml, double mu, double ms,
	uint32_t seed)
{
	nstars_ = n;
	sx_.alloc(n);
	sy_.alloc(n);
	sm_.alloc(n);
	k_generate_stars<<<blocks_for(n, 256), 256, 0, stream_>>>(sx_.ptr, sy_.ptr, sm_.ptr, n, rectangular, c_re, c_im, mf,
		ml, mu, ms, seed);
	MLENS_HIP_CHECK(hipGetLastError());
	MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
}

template <typename F>
__global__ void k_stars_aos(const double* sx, const double* sy, const double* sm, int n, F* out)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	out[3 * (long long)i] = F(sx[i]);
	out[3 * (long long)i + 1] = F(sy[i]);
	out[3 * (long long)i + 2] = F(sm[i]);
}

template <typename F>
void Engine::download_stars_as(F* aos)
{
	// in pieces, so that the rows' buffer stays small beside a large field (6 MB)
	constexpr int PIECE = 1 << 18;
	stars_aos_.alloc(3 * sizeof(F) * size_t(std::min(std::max(nstars_, 0), PIECE)));
	F* d = reinterpret_cast<F*>(stars_aos_.ptr);
	for (int i = 0; i < nstars_; i += std::min(PIECE, nstars_ - i))
	{
		const int n = std::min(PIECE, nstars_ - i);
		k_stars_aos<F><<<blocks_for(n, 256), 256, 0, stream_>>>(sx_.ptr + i, sy_.ptr + i, sm_.ptr + i, n, d);
		MLENS_HIP_CHECK(hipGetLastError());
		MLENS_HIP_CHECK(hipMemcpyAsync(aos + 3 * size_t(i), d, 3 * sizeof(F) * size_t(n), hipMemcpyDeviceToHost, stream_));
	}
	MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
}

void Engine::download_stars(double* aos) { download_stars_as(aos); }
void Engine::download_stars(float* aos) { download_stars_as(aos); }

/*
star.cuh:124-161: totals in FP64 over STAT_CHAINS interleaved chains (star i belongs to chain
i % STAT_CHAINS), each summed in order, then the chains by a tree. A block takes STAT_GROUP
chains, a lane per chain and sixteenth of a row of stars: the lanes fetch and take logarithms
side by side, then each chain's own lane adds its terms in order. One block walking all the chains
took 2.2 ms for 1.28e6 stars, the 16 blocks take 0.48.
*/
constexpr int STAT_CHAINS = 256;
constexpr int STAT_GROUP = 16;   // chains of a block: 128 bytes of consecutive stars
constexpr int STAT_ROWS = 16;    // stars of each chain in flight

__global__ __launch_bounds__(STAT_GROUP * STAT_ROWS) void k_star_chains(const double* __restrict__ sm, int n, double* __restrict__ part)
{
	__shared__ double m_s[STAT_ROWS][STAT_GROUP], log_s[STAT_ROWS][STAT_GROUP];
	const int c = threadIdx.x % STAT_GROUP, r = threadIdx.x / STAT_GROUP;
	const int chain = blockIdx.x * STAT_GROUP + c;
	double t = 0, t2 = 0, tl = 0, lo = 1e300, hi = -1e300;
	long long i = chain + (long long)r * STAT_CHAINS;
	double next = i < n ? sm[i] : 0.0;
	for (long long base = 0; base * STAT_CHAINS < n; base += STAT_ROWS)
	{
		const double m = next;
		i += (long long)STAT_ROWS * STAT_CHAINS;
		next = i < n ? sm[i] : 0.0;
		m_s[r][c] = m;
		log_s[r][c] = log(m);
		__syncthreads();
		if (r == 0)
		{
			for (int k = 0; k < STAT_ROWS && chain + (base + k) * STAT_CHAINS < n; k++)
			{
				const double v = m_s[k][c];
				t += v;
				t2 += v * v;
				tl += v * v * log_s[k][c];
				lo = fmin(lo, v);
				hi = fmax(hi, v);
			}
		}
		__syncthreads();
	}
	if (r != 0) return;
	part[chain] = t;
	part[STAT_CHAINS + chain] = t2;
	part[2 * STAT_CHAINS + chain] = tl;
	part[3 * STAT_CHAINS + chain] = lo;
	part[4 * STAT_CHAINS + chain] = hi;
}

__global__ __launch_bounds__(STAT_CHAINS) void k_star_stats(const double* __restrict__ part, double* out)
{
	__shared__ double s[5][STAT_CHAINS];
	const int k = threadIdx.x;
	for (int q = 0; q < 5; q++) s[q][k] = part[q * STAT_CHAINS + k];
	__syncthreads();
	for (int off = STAT_CHAINS / 2; off > 0; off >>= 1)
	{
		if (k < off)
		{
			for (int q = 0; q < 3; q++) s[q][k] += s[q][k + off];
			s[3][k] = fmin(s[3][k], s[3][k + off]);
			s[4][k] = fmax(s[4][k], s[4][k + off]);
		}
		__syncthreads();
	}
	if (k < 5) out[k] = s[k][0];
}

StarStats Engine::star_stats()
{
	scratch_d_.alloc(5 * STAT_CHAINS + 8);
	double* out = scratch_d_.ptr + 5 * STAT_CHAINS;
	k_star_chains<<<STAT_CHAINS / STAT_GROUP, STAT_GROUP * STAT_ROWS, 0, stream_>>>(sm_.ptr, nstars_, scratch_d_.ptr);
	k_star_stats<<<1, STAT_CHAINS, 0, stream_>>>(scratch_d_.ptr, out);
	MLENS_HIP_CHECK(hipGetLastError());
	double h[5];
	MLENS_HIP_CHECK(hipMemcpyAsync(h, out, sizeof(h), hipMemcpyDeviceToHost, stream_));
	MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
	return StarStats{h[0], h[1], h[2], h[3], h[4]};
}

/* ---------------------------------------------------------------------------
Exclusive scan of int4 records (three passes: tiles, tile totals, add-back).
out has n + 1 entries; out[n] is the grand total.
--------------------------------------------------------------------------- */
struct I4
{
	int x, y, z, w;
};
__device__ __forceinline__ I4 operator+(I4 a, I4 b) { return I4{a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w}; }
__device__ __forceinline__ I4 operator-(I4 a, I4 b) { return I4{a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w}; }
__device__ __forceinline__ int comp(I4 a, int q) { return q == 0 ? a.x : (q == 1 ? a.y : (q == 2 ? a.z : a.w)); }

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 4;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__device__ inline I4 block_exclusive_scan(I4 v, I4* s, I4& total)
{
	int t = threadIdx.x;
	s[t] = v;
	__syncthreads();
	for (int off = 1; off < SCAN_THREADS; off <<= 1)
	{
		I4 add = t >= off ? s[t - off] : I4{0, 0, 0, 0};
		__syncthreads();
		s[t] = s[t] + add;
		__syncthreads();
	}
	total = s[SCAN_THREADS - 1];
	I4 ex = t > 0 ? s[t - 1] : I4{0, 0, 0, 0};
	__syncthreads();
	return ex;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_tiles(const I4* in, I4* out, I4* tile_sums, int n)
{
	__shared__ I4 s[SCAN_THREADS];
	long long base = (long long)blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_ITEMS;
	I4 v[SCAN_ITEMS];
	I4 sum{0, 0, 0, 0};
#pragma unroll
	for (int k = 0; k < SCAN_ITEMS; k++)
	{
		v[k] = (base + k < n) ? in[base + k] : I4{0, 0, 0, 0};
		sum = sum + v[k];
	}
	I4 total;
	I4 run = block_exclusive_scan(sum, s, total);
#pragma unroll
	for (int k = 0; k < SCAN_ITEMS; k++)
	{
		if (base + k < n) out[base + k] = run;
		run = run + v[k];
	}
	if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_tile_sums(I4* tile_sums, int ntiles, I4* grand)
{
	__shared__ I4 s[SCAN_THREADS];
	I4 carry{0, 0, 0, 0};
	for (int base = 0; base < ntiles; base += SCAN_THREADS)
	{
		int i = base + threadIdx.x;
		I4 v = i < ntiles ? tile_sums[i] : I4{0, 0, 0, 0};
		I4 total;
		I4 ex = block_exclusive_scan(v, s, total);
		if (i < ntiles) tile_sums[i] = ex + carry;
		carry = carry + total;
	}
	if (threadIdx.x == 0) *grand = carry;
}

__global__ void k_scan_add(I4* out, const I4* tile_sums, int n, const I4* grand)
{
	long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) out[i] = out[i] + tile_sums[i / SCAN_TILE];
	if (i == n) out[n] = *grand;
}

static void scan_i4(const I4* in, I4* out, I4* tiles, int n, hipStream_t st)
{
	int ntiles = std::max(1, (n + SCAN_TILE - 1) / SCAN_TILE);
	k_scan_tiles<<<ntiles, SCAN_THREADS, 0, st>>>(in, out, tiles, n);
	k_scan_tile_sums<<<1, SCAN_THREADS, 0, st>>>(tiles, ntiles, tiles + ntiles);
	k_scan_add<<<blocks_for(n + 1, 256), 256, 0, st>>>(out, tiles, n, tiles + ntiles);
	MLENS_HIP_CHECK(hipGetLastError());
}

/* ---------------------------------------------------------------------------
Quadtree (tree_node.cuh:32-561, level loop of ipm.cuh:740-839)
--------------------------------------------------------------------------- */
struct TreeView
{
	double *cx, *cy, *hl;
	int *level, *parent, *child0, *begin, *count, *nnbr, *nm2l, *np2l, *nbr, *m2l, *p2l;
};

__device__ __forceinline__ int quadrant(double x, double y, double cx, double cy)   // tree_node.cuh:432-477
{
	if (y >= cy) return (x >= cx) ? 0 : 1;
	return (x < cx) ? 2 : 3;
}

// what the host reads after each level: nodes that split, and the stars of the largest of them
struct LevelCount
{
	int split, largest;
};

// The root (ipm.cuh:746-773): it splits when it holds more stars than a leaf may sum directly
// (tree_node.cuh:321-345).
__global__ void k_make_root(TreeView t, double half_length, int n, int* flags, int* rank, LevelCount* counts)
{
	t.cx[0] = 0;
	t.cy[0] = 0;
	t.hl[0] = half_length;
	t.level[0] = 0;
	t.parent[0] = -1;
	t.child0[0] = -1;
	t.begin[0] = 0;
	t.count[0] = n;
	t.nnbr[0] = 0;
	t.nm2l[0] = 0;
	t.np2l[0] = 0;
	flags[0] = n > MAX_NUM_STARS_DIRECT ? 1 : 0;
	rank[0] = 0;
	counts->split = flags[0];
	counts->largest = n;
}

// rank[i] = nodes before i that split; one block, for levels of at most RANK_MAX nodes. Clears
// nothing: k_set_neighbors left the largest count in counts.
constexpr int RANK_THREADS = 1024;
constexpr int RANK_MAX = 32768;

__global__ __launch_bounds__(RANK_THREADS) void k_rank(const int* __restrict__ flags, int* __restrict__ rank, int nl, LevelCount* counts)
{
	__shared__ int part[RANK_THREADS / 64];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	int carry = 0;
	for (int base = 0; base < nl; base += RANK_THREADS)
	{
		const int i = base + threadIdx.x;
		const int f = i < nl ? flags[i] : 0;
		const unsigned long long m = __ballot(f);
		if (lane == 0) part[wave] = __popcll(m);
		__syncthreads();
		int before = carry;
		for (int w = 0; w < RANK_THREADS / 64; w++)
		{
			if (w < wave) before += part[w];
			carry += part[w];
		}
		if (i < nl) rank[i] = before + int(__popcll(m & ((1ull << lane) - 1)));
		__syncthreads();
	}
	if (threadIdx.x == 0) counts->split = carry;
}

__global__ void k_flags_to_i4(const int* flags, I4* out, int nl)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < nl) out[i] = I4{flags[i], 0, 0, 0};
}

__global__ void k_i4_to_rank(const I4* in, int* rank, int nl, LevelCount* counts)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < nl) rank[i] = in[i].x;
	if (i == nl) counts->split = in[nl].x;
}

// child q of node i (tree_node.cuh:151-177: offsets (+,+), (-,+), (-,-), (+,-))
__device__ __forceinline__ void make_child(TreeView t, int i, int c0, int q)
{
	const double nh = t.hl[i] / 2;
	const double ox = (q == 0 || q == 3) ? 1 : -1, oy = q < 2 ? 1 : -1;
	const int c = c0 + q;
	t.cx[c] = t.cx[i] + nh * ox;
	t.cy[c] = t.cy[i] + nh * oy;
	t.hl[c] = nh;
	t.level[c] = t.level[i] + 1;
	t.parent[c] = i;
	t.child0[c] = -1;
}

/*
A level's splits, one block per node: its four children, and a stable partition of its stars into
them (sort_stars_kernel, tree_node.cuh:392-501) by way of the scratch arrays. One launch per level
where the device-wide partition below takes seven; that one is kept for nodes of more than
SPLIT_MAX stars, whose passes a single block would walk alone.
*/
constexpr int SPLIT_MAX = 16384;

// A node of a level that splits further: its place in the leaf tables, -1 for one that splits itself. leaf0 leaves stand
// on earlier levels; build_leaf_tables numbers the last level, whose nodes are all leaves.
__device__ __forceinline__ int leaf_index(const int* flags, const int* rank, int k, int leaf0) { return flags[k] ? -1 : leaf0 + k - rank[k]; }

template <int THREADS>
__global__ __launch_bounds__(THREADS) void k_split_nodes(TreeView t, int l0, const int* __restrict__ flags, const int* __restrict__ rank,
	int base, int leaf0, int* __restrict__ leaf_of_node, double* sx, double* sy, double* sm, double* tx, double* ty, double* tm)
{
	constexpr int WAVES = THREADS / 64;
	__shared__ int part[4][WAVES];
	const int i = l0 + blockIdx.x;
	if (threadIdx.x == 0) leaf_of_node[i] = leaf_index(flags, rank, blockIdx.x, leaf0);
	if (!flags[blockIdx.x]) return;
	const int c0 = base + 4 * rank[blockIdx.x];
	const int b = t.begin[i], n = t.count[i];
	const double cx = t.cx[i], cy = t.cy[i];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	// quadrant sizes
	int mine[4] = {0, 0, 0, 0};
	for (int s = threadIdx.x; s < n; s += THREADS)
	{
		const int q = quadrant(sx[b + s], sy[b + s], cx, cy);
#pragma unroll
		for (int k = 0; k < 4; k++) mine[k] += q == k;
	}
#pragma unroll
	for (int k = 0; k < 4; k++)
	{
		for (int off = 32; off > 0; off >>= 1) mine[k] += __shfl_xor(mine[k], off);
		if (lane == 0) part[k][wave] = mine[k];
	}
	__syncthreads();
	int start[4], total = 0;
#pragma unroll
	for (int k = 0; k < 4; k++)
	{
		int c = 0;
		for (int w = 0; w < WAVES; w++) c += part[k][w];
		start[k] = b + total;
		total += c;
		mine[k] = c;
	}
	if (threadIdx.x == 0) t.child0[i] = c0;
	if (threadIdx.x < 4)
	{
		const int q = threadIdx.x;
		make_child(t, i, c0, q);
		t.begin[c0 + q] = q == 0 ? start[0] : (q == 1 ? start[1] : (q == 2 ? start[2] : start[3]));
		t.count[c0 + q] = q == 0 ? mine[0] : (q == 1 ? mine[1] : (q == 2 ? mine[2] : mine[3]));
	}
	// stable placement, THREADS stars at a time
	for (int s0 = 0; s0 < n; s0 += THREADS)
	{
		__syncthreads();
		const int s = s0 + threadIdx.x;
		double x = 0, y = 0, m = 0;
		int q = 4;
		if (s < n)
		{
			x = sx[b + s];
			y = sy[b + s];
			m = sm[b + s];
			q = quadrant(x, y, cx, cy);
		}
		int before = 0;
#pragma unroll
		for (int k = 0; k < 4; k++)
		{
			const unsigned long long mk = __ballot(q == k);
			if (lane == 0) part[k][wave] = __popcll(mk);
			if (q == k) before = __popcll(mk & ((1ull << lane) - 1));
		}
		__syncthreads();
#pragma unroll
		for (int k = 0; k < 4; k++)
		{
			int all = 0, ahead = 0;
			for (int w = 0; w < WAVES; w++)
			{
				if (w < wave) ahead += part[k][w];
				all += part[k][w];
			}
			if (q == k)
			{
				const int dst = start[k] + ahead + before;
				tx[dst] = x;
				ty[dst] = y;
				tm[dst] = m;
			}
			start[k] += all;
		}
	}
	__syncthreads();
	for (int s = threadIdx.x; s < n; s += THREADS)
	{
		sx[b + s] = tx[b + s];
		sy[b + s] = ty[b + s];
		sm[b + s] = tm[b + s];
	}
}

// the device-wide partition of a level (k_split_nodes takes the levels whose nodes are small)
__global__ void k_make_children(TreeView t, int l0, int l1, const int* flags, const int* rank, int base, int leaf0, int* leaf_of_node)
{
	int i = l0 + blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= l1) return;
	leaf_of_node[i] = leaf_index(flags, rank, i - l0, leaf0);
	if (!flags[i - l0]) return;
	int c0 = base + 4 * rank[i - l0];
	t.child0[i] = c0;
	for (int q = 0; q < 4; q++) make_child(t, i, c0, q);
}

__global__ void k_star_onehot(TreeView t, const double* sx, const double* sy, const int* star_node, int l0,
	const int* flags, I4* onehot, int n)
{
	int s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= n) return;
	int node = star_node[s];
	I4 v{0, 0, 0, 0};
	if (node >= 0 && flags[node - l0])
	{
		int q = quadrant(sx[s], sy[s], t.cx[node], t.cy[node]);
		v.x = q == 0;
		v.y = q == 1;
		v.z = q == 2;
		v.w = q == 3;
	}
	onehot[s] = v;
}

__global__ void k_child_ranges(TreeView t, int l0, int l1, const int* flags, const I4* pre)
{
	int i = l0 + blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= l1 || !flags[i - l0]) return;
	int b = t.begin[i];
	I4 c = pre[b + t.count[i]] - pre[b];
	int c0 = t.child0[i];
	int start = b;
	for (int q = 0; q < 4; q++)
	{
		int cq = comp(c, q);
		t.begin[c0 + q] = start;
		t.count[c0 + q] = cq;
		start += cq;
	}
}

// stable partition of each split node's stars into its four children (sort_stars_kernel, tree_node.cuh:392-501)
__global__ void k_star_scatter(TreeView t, const double* sx, const double* sy, const double* sm, double* tx, double* ty,
	double* tm, const int* star_node, int* star_node_out, int l0, const int* flags, const I4* pre, int n)
{
	int s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= n) return;
	int node = star_node[s];
	if (node >= 0 && flags[node - l0])
	{
		int q = quadrant(sx[s], sy[s], t.cx[node], t.cy[node]);
		int b = t.begin[node];
		int rank = comp(pre[s], q) - comp(pre[b], q);
		int child = t.child0[node] + q;
		int dst = t.begin[child] + rank;
		tx[dst] = sx[s];
		ty[dst] = sy[s];
		tm[dst] = sm[s];
		star_node_out[dst] = child;
	}
	else
	{
		tx[s] = sx[s];
		ty[s] = sy[s];
		tm[s] = sm[s];
		star_node_out[s] = -1;   // star now sits in a leaf
	}
}

/*
The lists of a level's nodes (tree_node.cuh:183-267) and the nodes that split next (the stars of a
node and its neighbours, 321-345). One wave per node, one candidate per lane: the four siblings, then
the four children of each neighbour of the parent (or that neighbour itself, where it is a leaf), in
the order the lists keep. A lane's place in its list is the number of lanes before it that chose the
same list. Walked by one lane per node, the candidates' dependent loads took 17 us a level.
*/
__global__ __launch_bounds__(256) void k_set_neighbors(TreeView t, int n0, int n1, int* flags, LevelCount* counts)
{
	const int i = n0 + blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
	if (i >= n1) return;
	const int par = t.parent[i];
	const double cx = t.cx[i], cy = t.cy[i], h = t.hl[i];
	enum
	{
		NONE,
		NEAR,
		M2L,
		P2L
	};
	int kind = NONE, c = -1, count = 0;
	if (lane < 4)
	{
		c = t.child0[par] + lane;
		count = t.count[c];
		if (count != 0 && c != i) kind = NEAR;
	}
	else if (lane < 4 + 4 * MAX_NUM_NEIGHBORS)
	{
		const int j = (lane - 4) >> 2, q = lane & 3;
		if (j < t.nnbr[par])
		{
			const int nb = t.nbr[8 * par + j];
			const int c0 = t.child0[nb];
			const bool leaf = c0 < 0;
			c = leaf ? nb : c0 + q;
			count = t.count[c];
			if (leaf)
			{
				if (q == 0 && count != 0) kind = (fabs(t.cx[c] - cx) < 3.5 * h && fabs(t.cy[c] - cy) < 3.5 * h) ? NEAR : P2L;
			}
			else if (count != 0)
				kind = (fabs(t.cx[c] - cx) < 3 * h && fabs(t.cy[c] - cy) < 3 * h) ? NEAR : M2L;
		}
	}
	const unsigned long long below = (1ull << lane) - 1;
	const unsigned long long near = __ballot(kind == NEAR), m2l = __ballot(kind == M2L), p2l = __ballot(kind == P2L);
	if (kind == NEAR) t.nbr[8 * (long long)i + __popcll(near & below)] = c;
	if (kind == M2L) t.m2l[27 * (long long)i + __popcll(m2l & below)] = c;
	if (kind == P2L) t.p2l[5 * (long long)i + __popcll(p2l & below)] = c;
	int stars = kind == NEAR ? count : 0;
	for (int off = 32; off > 0; off >>= 1) stars += __shfl_xor(stars, off);
	if (lane == 0)
	{
		t.nnbr[i] = __popcll(near);
		t.nm2l[i] = __popcll(m2l);
		t.np2l[i] = __popcll(p2l);
		const int own = t.count[i];
		const bool split = stars + own > MAX_NUM_STARS_DIRECT;
		flags[i - n0] = split;
		// few nodes raise the maximum: most need no atomic on the one address
		if (split && own > *static_cast<volatile int*>(&counts->largest)) atomicMax(&counts->largest, own);
	}
}

template <typename T>
static void grow(DeviceBuffer<T>& b, size_t used, size_t n)
{
	if (n <= b.count) return;
	T* p = nullptr;
	MLENS_HIP_CHECK(hipMalloc(&p, n * sizeof(T)));
	if (used) MLENS_HIP_CHECK(hipMemcpy(p, b.ptr, used * sizeof(T), hipMemcpyDeviceToDevice));
	b.free();
	b.ptr = p;
	b.count = n;
}

void Engine::ensure_node_capacity(int n)
{
	if (n <= node_cap_) return;
	int cap = std::max(n, std::max(1024, 2 * node_cap_));
	size_t u = size_t(num_nodes_);
	grow(ncx_, u, cap);
	grow(ncy_, u, cap);
	grow(nhl_, u, cap);
	grow(nlevel_, u, cap);
	grow(nparent_, u, cap);
	grow(nchild0_, u, cap);
	grow(nbegin_, u, cap);
	grow(ncount_, u, cap);
	grow(nnnbr_, u, cap);
	grow(nnm2l_, u, cap);
	grow(nnp2l_, u, cap);
	grow(nnbr_, u * 8, size_t(cap) * 8);
	grow(nm2l_, u * 27, size_t(cap) * 27);
	grow(np2l_, u * 5, size_t(cap) * 5);
	grow(leaf_of_node_, u, cap);
	node_cap_ = cap;
}

static TreeView view(DeviceBuffer<double>& cx, DeviceBuffer<double>& cy, DeviceBuffer<double>& hl, DeviceBuffer<int>& lv,
	DeviceBuffer<int>& par, DeviceBuffer<int>& c0, DeviceBuffer<int>& b, DeviceBuffer<int>& n, DeviceBuffer<int>& nn,
	DeviceBuffer<int>& nm, DeviceBuffer<int>& np, DeviceBuffer<int>& nb, DeviceBuffer<int>& m2l, DeviceBuffer<int>& p2l)
{
	return TreeView{cx.ptr, cy.ptr, hl.ptr, lv.ptr, par.ptr, c0.ptr, b.ptr, n.ptr, nn.ptr, nm.ptr, np.ptr, nb.ptr, m2l.ptr, p2l.ptr};
}

void Engine::build_tree(double root_half_length)
{
	const int n = nstars_;
	num_nodes_ = 0;
	// an even field ends with 0.6 to 0.9 nodes per star; growing copies every node array (0.15 ms each time at 7e3 stars)
	ensure_node_capacity(std::max(1024, n + n / 8));
	level_start_.assign({0, 1});
	levels_ = 0;
	num_leaves_ = 0;   // on the levels before this one

	num_nodes_ = 1;
	const size_t ns = size_t(std::max(n, 1));
	tx_.alloc(ns);
	ty_.alloc(ns);
	tm_.alloc(ns);
	level_count_.alloc(2);
	LevelCount* counts = reinterpret_cast<LevelCount*>(level_count_.ptr);
	auto tree = [&]() {
		return view(ncx_, ncy_, nhl_, nlevel_, nparent_, nchild0_, nbegin_, ncount_, nnnbr_, nnm2l_, nnp2l_, nnbr_, nm2l_, np2l_);
	};
	node_flag_.alloc(node_cap_);
	node_rank_.alloc(node_cap_);
	k_make_root<<<1, 1, 0, stream_>>>(tree(), root_half_length, n, node_flag_.ptr, node_rank_.ptr, counts);
	MLENS_HIP_CHECK(hipGetLastError());
	// the device-wide partition's scratch, taken only if a level needs it
	DeviceBuffer<char> sbuf;
	bool star_nodes = false;   // star_node_ holds every star's node of this level (-1: in a leaf)
	while (true)
	{
		const int l0 = level_start_[levels_], l1 = level_start_[levels_ + 1], nl = l1 - l0;
		const size_t tiles_n = 2 * (size_t(std::max(n, nl)) / SCAN_TILE + 4);
		if (nl > RANK_MAX)
		{
			sbuf.alloc(sizeof(I4) * (2 * size_t(nl) + 1 + tiles_n));
			I4* f = reinterpret_cast<I4*>(sbuf.ptr);
			I4* r = f + nl;
			k_flags_to_i4<<<blocks_for(nl, 256), 256, 0, stream_>>>(node_flag_.ptr, f, nl);
			scan_i4(f, r, r + nl + 1, nl, stream_);
			k_i4_to_rank<<<blocks_for(nl + 1, 256), 256, 0, stream_>>>(r, node_rank_.ptr, nl, counts);
		}
		else if (levels_ > 0)
			k_rank<<<1, RANK_THREADS, 0, stream_>>>(node_flag_.ptr, node_rank_.ptr, nl, counts);
		MLENS_HIP_CHECK(hipGetLastError());
		LevelCount lc;
		MLENS_HIP_CHECK(hipMemcpyAsync(&lc, counts, sizeof(lc), hipMemcpyDeviceToHost, stream_));
		MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
		if (lc.split == 0)
		{
			last_level_leaf0_ = num_leaves_;
			num_leaves_ += nl;
			break;
		}
		const int base = l1;
		ensure_node_capacity(base + 4 * lc.split);
		const TreeView t = tree();
		if (lc.largest > SPLIT_MAX)
		{
			sbuf.alloc(sizeof(I4) * (2 * size_t(n) + 1 + tiles_n));
			I4* onehot = reinterpret_cast<I4*>(sbuf.ptr);
			I4* pre = onehot + n;
			I4* tiles = pre + n + 1;
			star_node_.alloc(ns);
			star_node_tmp_.alloc(ns);
			if (!star_nodes) MLENS_HIP_CHECK(hipMemsetAsync(star_node_.ptr, 0, ns * sizeof(int), stream_));
			star_nodes = true;
			k_make_children<<<blocks_for(nl, 256), 256, 0, stream_>>>(t, l0, l1, node_flag_.ptr, node_rank_.ptr, base,
				num_leaves_, leaf_of_node_.ptr);
			k_star_onehot<<<blocks_for(n, 256), 256, 0, stream_>>>(t, sx_.ptr, sy_.ptr, star_node_.ptr, l0, node_flag_.ptr, onehot, n);
			MLENS_HIP_CHECK(hipGetLastError());
			scan_i4(onehot, pre, tiles, n, stream_);
			k_child_ranges<<<blocks_for(nl, 256), 256, 0, stream_>>>(t, l0, l1, node_flag_.ptr, pre);
			k_star_scatter<<<blocks_for(n, 256), 256, 0, stream_>>>(t, sx_.ptr, sy_.ptr, sm_.ptr, tx_.ptr, ty_.ptr, tm_.ptr,
				star_node_.ptr, star_node_tmp_.ptr, l0, node_flag_.ptr, pre, n);
			MLENS_HIP_CHECK(hipGetLastError());
			std::swap(sx_.ptr, tx_.ptr);
			std::swap(sy_.ptr, ty_.ptr);
			std::swap(sm_.ptr, tm_.ptr);
			std::swap(sx_.count, tx_.count);
			std::swap(sy_.count, ty_.count);
			std::swap(sm_.count, tm_.count);
			std::swap(star_node_.ptr, star_node_tmp_.ptr);
			std::swap(star_node_.count, star_node_tmp_.count);
		}
		else
		{
			// a block per node, as wide as its largest node can use (children never hold more stars than
			// their parent, so the device-wide partition is not needed again)
			auto split = [&](auto kernel, int threads) {
				kernel<<<nl, threads, 0, stream_>>>(t, l0, node_flag_.ptr, node_rank_.ptr, base, num_leaves_, leaf_of_node_.ptr, sx_.ptr,
					sy_.ptr, sm_.ptr, tx_.ptr, ty_.ptr, tm_.ptr);
			};
			if (lc.largest <= 256) split(k_split_nodes<64>, 64);
			else if (lc.largest <= 2048) split(k_split_nodes<256>, 256);
			else split(k_split_nodes<1024>, 1024);
			MLENS_HIP_CHECK(hipGetLastError());
		}
		num_leaves_ += nl - lc.split;
		num_nodes_ = base + 4 * lc.split;
		levels_++;
		level_start_.push_back(num_nodes_);
		node_flag_.alloc(4 * size_t(lc.split));
		node_rank_.alloc(4 * size_t(lc.split));
		MLENS_HIP_CHECK(hipMemsetAsync(counts, 0, sizeof(LevelCount), stream_));
		k_set_neighbors<<<blocks_for(4 * lc.split, 4), 256, 0, stream_>>>(t, base, num_nodes_, node_flag_.ptr, counts);
		MLENS_HIP_CHECK(hipGetLastError());
	}
}

void Engine::export_tree(double* geom, int* info, int* lists) const
{
	int nn = num_nodes_;
	std::vector<double> cx(nn), cy(nn), hl(nn);
	std::vector<int> lv(nn), par(nn), c0(nn), b(nn), n(nn), nnb(nn), nm(nn), np(nn), nb(size_t(nn) * 8), m2l(size_t(nn) * 27),
		p2l(size_t(nn) * 5);
	auto get = [](auto& v, const auto& d, size_t cnt) {
		MLENS_HIP_CHECK(hipMemcpy(v.data(), d.ptr, cnt * sizeof(v[0]), hipMemcpyDeviceToHost));
	};
	get(cx, ncx_, nn);
	get(cy, ncy_, nn);
	get(hl, nhl_, nn);
	get(lv, nlevel_, nn);
	get(par, nparent_, nn);
	get(c0, nchild0_, nn);
	get(b, nbegin_, nn);
	get(n, ncount_, nn);
	get(nnb, nnnbr_, nn);
	get(nm, nnm2l_, nn);
	get(np, nnp2l_, nn);
	get(nb, nnbr_, size_t(nn) * 8);
	get(m2l, nm2l_, size_t(nn) * 27);
	get(p2l, np2l_, size_t(nn) * 5);
	for (int i = 0; i < nn; i++)
	{
		geom[3 * i] = cx[i];
		geom[3 * i + 1] = cy[i];
		geom[3 * i + 2] = hl[i];
		int* f = info + 9 * i;
		f[0] = lv[i];
		f[1] = par[i];
		f[2] = c0[i];
		f[3] = c0[i] >= 0 ? 4 : 0;
		f[4] = b[i];
		f[5] = n[i];
		f[6] = nnb[i];
		f[7] = nm[i];
		f[8] = np[i];
		int* L = lists + 40 * i;
		for (int j = 0; j < 40; j++) L[j] = -1;
		for (int j = 0; j < nnb[i]; j++) L[j] = nb[8 * size_t(i) + j];
		for (int j = 0; j < nm[i]; j++) L[8 + j] = m2l[27 * size_t(i) + j];
		for (int j = 0; j < np[i]; j++) L[35 + j] = p2l[5 * size_t(i) + j];
	}
}

/* ---------------------------------------------------------------------------
FMM in node-normalised units (fmm.cuh:21-464). One thread per (node, order).
Binomial coefficients are exact integers rounded once to double; the
reference's int32 table wraps for rows >= 34 (binomial_coefficients.cuh:11-44).
--------------------------------------------------------------------------- */
__device__ __forceinline__ double binom(const double* B, int n, int k)
{
	return (n < k) ? 0.0 : B[n * (n + 1) / 2 + k];
}

__device__ __forceinline__ dcx ld(const double* a, long long i) { return dcx{a[2 * i], a[2 * i + 1]}; }
__device__ __forceinline__ void st(double* a, long long i, dcx v)
{
	a[2 * i] = v.re;
	a[2 * i + 1] = v.im;
}

// P2M at every leaf, zero where it holds no stars (fmm.cuh:21-98); M2M writes the other nodes
__global__ void k_p2m(TreeView t, int nn, int p, const double* sx, const double* sy, const double* sm, double* mult)
{
	long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	int i = int(g / (p + 1));
	int k = int(g % (p + 1));
	if (i >= nn) return;
	if (t.child0[i] >= 0) return;
	double cx = t.cx[i], cy = t.cy[i], h = t.hl[i];
	int b = t.begin[i], n = t.count[i];
	dcx r = {0, 0};
	if (k == 0)
	{
		for (int s = b; s < b + n; s++) r.re += sm[s];
	}
	else
	{
		for (int s = b; s < b + n; s++)
		{
			dcx dz = dcx{(sx[s] - cx) / h, (sy[s] - cy) / h};
			dcx pw = dev::cpow(dz, k);
			r = dev::sub(r, dev::scale(pw, sm[s]));
		}
		r = dev::scale(r, 1.0 / k);
	}
	st(mult, (long long)i * (p + 1) + k, r);
}

/*
M2M, children to parent (fmm.cuh:109-192): one thread per (child, order), the four children of a
parent summed in order. Blocks hold whole sibling groups, FMM_THREADS / (p + 1) children rounded down
to groups; their multipoles and the binomials come from LDS, since every order's chain of steps
reads all of them (a level took 16 us with one thread per parent and order and the operands in L2).
*/
constexpr int FMM_THREADS = 256;
constexpr int FMM_BINOMIALS = (MAX_EXPANSION_ORDER + 1) * (MAX_EXPANSION_ORDER + 2) / 2;   // rows 0..p

__host__ __device__ inline int fmm_nodes_per_block(int p) { return FMM_THREADS / (p + 1) / 4 * 4; }

__global__ __launch_bounds__(FMM_THREADS) void k_m2m(TreeView t, int c0, int c1, int p, const double* __restrict__ B, double* mult)
{
	__shared__ dcx m[FMM_THREADS], part[FMM_THREADS];
	__shared__ double b[FMM_BINOMIALS];
	const int P = p + 1, per = fmm_nodes_per_block(p);
	const int first = c0 + blockIdx.x * per, n = min(per, c1 - first);
	const int x = threadIdx.x, ci = x / P, l = x - ci * P;
	for (int i = x; i < p * (p + 1) / 2; i += FMM_THREADS) b[i] = B[i];
	const bool on = ci < n;
	if (on) m[x] = ld(mult, (long long)first * P + x);
	__syncthreads();
	const int c = first + ci;
	int par = 0;
	if (on)
	{
		par = t.parent[c];
		const dcx* mc = m + ci * P;
		dcx r = mc[0];
		if (l > 0)
		{
			dcx dz = dcx{(t.cx[c] - t.cx[par]) / t.hl[c], (t.cy[c] - t.cy[par]) / t.hl[c]};
			dcx idz = dev::cdiv(dcx{1, 0}, dz);
			r = dcx{0, 0};
			const double* row = b + (l - 1) * l / 2;   // C(l - 1, .)
			for (int k = l; k >= 1; k--)
			{
				r = dev::add(r, dev::scale(mc[k], row[k - 1]));
				r = dev::mul(r, idz);
			}
			r = dev::sub(r, dev::scale(mc[0], 1.0 / l));
			r = dev::mul(r, dev::cpow(dz, l));
			r = dev::scale(r, ldexp(1.0, -l));
		}
		part[x] = r;
	}
	__syncthreads();
	if (!on || (ci & 3) != 0) return;
	dcx acc = {0, 0};
	for (int q = 0; q < 4; q++) acc = dev::add(acc, part[x + q * P]);
	st(mult, (long long)par * P + l, acc);
}

// L2L, M2L and P2L for one level (fmm.cuh:204-464). The M2L sums are recurrences here (do_m2l) or
// were left in local by k_m2l.
// Blocks as in k_m2m, their parents' expansions and the binomials in LDS.
__global__ __launch_bounds__(FMM_THREADS) void k_local(TreeView t, int l0, int l1, int p, const double* __restrict__ B,
	const double* __restrict__ mult, double* local, const double* __restrict__ sx, const double* __restrict__ sy,
	const double* __restrict__ sm, int do_m2l)
{
	__shared__ dcx pl[FMM_THREADS / 4];
	__shared__ double b[FMM_BINOMIALS];
	const int P = p + 1, per = fmm_nodes_per_block(p);
	const int first = l0 + blockIdx.x * per, n = min(per, l1 - first);
	const int x = threadIdx.x, ci = x / P, l = x - ci * P;
	for (int k = x; k < P * (P + 1) / 2; k += FMM_THREADS) b[k] = B[k];
	if (x < n / 4 * P) pl[x] = ld(local, (long long)t.parent[first + 4 * (x / P)] * P + x % P);
	__syncthreads();
	if (ci >= n) return;
	const int i = first + ci;
	const double cx = t.cx[i], cy = t.cy[i], h = t.hl[i];
	dcx acc;
	{
		int par = t.parent[i];
		const dcx* lp = pl + (ci >> 2) * P;
		dcx dz = dcx{(cx - t.cx[par]) / t.hl[par], (cy - t.cy[par]) / t.hl[par]};
		dcx r = {0, 0};
		for (int k = p; k >= 1; k--)
		{
			r = dev::add(r, dev::scale(lp[k], k < l ? 0.0 : b[k * (k + 1) / 2 + l]));
			r = dev::mul(r, dz);
		}
		r = dev::cdiv(r, dev::cpow(dz, l));
		acc = dev::scale(r, ldexp(1.0, -l));
	}
	for (int j = 0; j < (do_m2l ? t.nm2l[i] : 0); j++)
	{
		int f = t.m2l[27 * i + j];
		const long long fb = (long long)f * (p + 1);
		double hf = t.hl[f];
		dcx dz = dcx{(t.cx[f] - cx) / hf, (t.cy[f] - cy) / hf};
		dcx mdz = dcx{-dz.re, -dz.im};
		dcx imdz = dev::cdiv(dcx{1, 0}, mdz);
		dcx b0 = ld(mult, fb);
		dcx r = {0, 0};
		if (l == 0)
		{
			for (int k = p; k >= 1; k--) r = dev::mul(dev::add(r, ld(mult, fb + k)), imdz);
			r = dev::add(r, dev::mul(b0, dev::clog(mdz)));
			r = dev::add(r, dev::scale(b0, log(hf)));
		}
		else
		{
			for (int k = p; k >= 1; k--) r = dev::mul(dev::add(r, dev::scale(ld(mult, fb + k), binom(B, l + k - 1, k - 1))), imdz);
			r = dev::sub(r, dev::scale(b0, 1.0 / l));
			r = dev::cdiv(r, dev::cpow(dz, l));
		}
		acc = dev::add(acc, r);
	}
	for (int j = 0; j < t.np2l[i]; j++)
	{
		int f = t.p2l[5 * i + j];
		for (int s = t.begin[f]; s < t.begin[f] + t.count[f]; s++)
		{
			dcx dz = dcx{(sx[s] - cx) / h, (sy[s] - cy) / h};
			double m = sm[s];
			if (l == 0)
			{
				acc = dev::add(acc, dev::scale(dev::clog(dcx{-dz.re, -dz.im}), m));
				acc.re += m * log(h);
			}
			else
			{
				acc = dev::sub(acc, dev::cdiv(dcx{m, 0}, dev::scale(dev::cpow(dz, l), double(l))));
			}
		}
	}
	if (!do_m2l) acc = dev::add(acc, ld(local, (long long)i * (p + 1) + l));
	st(local, (long long)i * (p + 1) + l, acc);
}

/*
Leaf tables for shooting: geometry, the near-field star list (own stars then
each neighbour's, alpha_star.cuh:26-37) and the deflection polynomial
A_i = (theta^2/h) i c_i of alpha_local.cuh:18-36, so that
alpha_local(z) = conj( sum_{i=1..p} A_i dz^(i-1) ), dz = (z - c)/h.
Leaves are numbered as the levels are split (leaf_index), the last level's nodes,
from `last` on, here: no scan over the nodes. 32 lanes per node, a near star and a
polynomial entry each: one lane per leaf wrote 2 KB in 24-byte steps (2.0 ms for
the 1.28e6-star tree).
*/
__global__ __launch_bounds__(256) void k_leaf_tables(TreeView t, int nn, int last, int last_leaf0, int p, double theta2, const double* __restrict__ sx,
	const double* __restrict__ sy, const double* __restrict__ sm, const double* __restrict__ local, int* leaf_of_node, double* geom,
	int* near_n, int* near_true, double* near_d, float* near_f, double* poly_d, float* poly_f)
{
	constexpr int LANES = 32;   // per leaf
	static_assert(MAX_NUM_STARS_DIRECT == LANES, "a lane per near star");
	static_assert((MAX_EXPANSION_ORDER + 3) / 4 * 4 <= LANES, "a lane per polynomial entry");
	__shared__ double lead_s[256 / LANES][LANES];
	const int lane = threadIdx.x % LANES, slot = threadIdx.x / LANES;
	const int i = blockIdx.x * (256 / LANES) + slot;
	const long long L = i >= nn ? -1 : (i >= last ? last_leaf0 + (i - last) : leaf_of_node[i]);
	const bool leaf = L >= 0;
	if (leaf && i >= last && lane == 0) leaf_of_node[i] = int(L);
	double cx = 0, cy = 0, h = 1, scale_l1 = 0, lead = 0;
	int total = 0, padded = 0;
	const int SD = poly_stride_d(p), SF = poly_stride_f(p);
	if (leaf)
	{
		cx = t.cx[i];
		cy = t.cy[i];
		h = t.hl[i];
		if (lane < 4) geom[4 * L + lane] = lane == 0 ? cx : (lane == 1 ? cy : (lane == 2 ? h : 1.0 / h));
		// near star `lane`: own stars, then each neighbour's, at most MAX_NUM_STARS_DIRECT
		int star = -1;
		const int nb = t.nnbr[i];
		for (int j = -1; j < nb; j++)
		{
			const int f = j < 0 ? i : t.nbr[8 * (long long)i + j];
			const int c = t.count[f];
			if (lane >= total && lane < total + c) star = t.begin[f] + (lane - total);
			total += c;
		}
		total = min(total, MAX_NUM_STARS_DIRECT);
		padded = (total + 3) & ~3;
		if (lane < padded)
		{
			// padding: massless stars far away (their terms are exactly 0)
			const bool real = lane < total;
			const double x = real ? sx[star] : 1e150, y = real ? sy[star] : 1e150, m = real ? sm[star] : 0.0;
			double* d = near_d + (L * MAX_NUM_STARS_DIRECT + lane) * 3;
			d[0] = x;
			d[1] = y;
			d[2] = m;
			float4 f = make_float4(1e18f, 1e18f, 0.0f, 0.0f);
			if (real) f = make_float4(float(x - cx), float(y - cy), float(m), 0.0f);
			reinterpret_cast<float4*>(near_f)[L * MAX_NUM_STARS_DIRECT + lane] = f;
		}
		// polynomial tables in descending degree, zero-padded at the top to a
		// multiple of 4: entry j of the FP64 table is the coefficient of
		// dz^(SD-1-j) in P(dz) = sum_{i=1..p} A_i dz^(i-1); entry j of the FP32
		// table is the coefficient of dz^(SF-1-j) in Q(dz) = sum_{i=2..p} A_i dz^(i-2)
		const long long lb = (long long)i * (p + 1);
		if (lane < SD)
		{
			const int q = SD - lane;   // A_q
			const dcx a = (q <= p) ? dev::scale(ld(local, lb + q), theta2 / h * q) : dcx{0, 0};
			poly_d[2 * (L * SD + lane)] = a.re;
			poly_d[2 * (L * SD + lane) + 1] = a.im;
		}
		// the FP32 evaluation skips its leading groups of 4 entries while their
		// terms together stay below 2^-28 of the scale of all terms, bounded over
		// the leaf (|dz| <= sqrt(2) in units of the half-size): an eighth of one
		// rounding of the FP32 sum, which carries about SF such roundings already.
		// On the 10000^2 map (p = 30) this leaves the mixed map's error against FP64
		// as it was (median 2.1e-6, max 6.9e-4) and takes 1% off the shot; at 2^-25
		// single pixels moved by 3e-3.
		scale_l1 = dev::cabs(dev::scale(ld(local, lb + 1), theta2 / h));
		if (lane < SF)
		{
			const int q = SF - lane + 1;   // A_q
			const dcx a = (q <= p && q >= 2) ? dev::scale(ld(local, lb + q), theta2 / h * q) : dcx{0, 0};
			poly_f[2 * (L * SF + lane)] = float(a.re);
			poly_f[2 * (L * SF + lane) + 1] = float(a.im);
			lead = dev::cabs(a) * pow(1.4143, double(q - 1));   // bound of A_q dz^(q-1) over the leaf
		}
	}
	lead_s[slot][lane] = lead;
	__syncthreads();
	if (!leaf || lane != 0) return;
	near_true[L] = total;
	double S = scale_l1, tail = 0;
	for (int j = 0; j < SF; j++) S += lead_s[slot][j];
	int skip = 0;
	for (int j0 = 0; j0 + 4 <= SF; j0 += 4)
	{
		const double* l = lead_s[slot] + j0;
		tail += l[0] + l[1] + l[2] + l[3];
		if (!(tail <= 0x1p-28 * S)) break;
		skip = j0 + 4;
	}
	near_n[L] = padded | (skip << 16);
}

void Engine::fmm(int p, const LensParams& lens)
{
	p_ = p;
	// exact Pascal triangle rows 0..2p (C(62, 31) < 2^64)
	{
		int nmax = 2 * p;
		std::vector<double> B(size_t(nmax + 1) * (nmax + 2) / 2);
		std::vector<unsigned long long> row(nmax + 1), prev(nmax + 1);
		for (int nr = 0; nr <= nmax; nr++)
		{
			for (int k = 0; k <= nr; k++) row[k] = (k == 0 || k == nr) ? 1ull : prev[k - 1] + prev[k];
			for (int k = 0; k <= nr; k++) B[size_t(nr) * (nr + 1) / 2 + k] = double(row[k]);
			prev = row;
		}
		binom_.alloc(B.size());
		MLENS_HIP_CHECK(hipMemcpy(binom_.ptr, B.data(), B.size() * sizeof(double), hipMemcpyHostToDevice));
	}
	const size_t nc = size_t(num_nodes_) * (p + 1) * 2;
	mult_.alloc(nc);
	local_.alloc(nc);
	// levels 0 and 1 have no far field; k_m2l or k_local writes the others
	const int far = levels_ >= 2 ? level_start_[2] : num_nodes_;
	MLENS_HIP_CHECK(hipMemsetAsync(local_.ptr, 0, size_t(far) * (p + 1) * 2 * sizeof(double), stream_));
	TreeView t = view(ncx_, ncy_, nhl_, nlevel_, nparent_, nchild0_, nbegin_, ncount_, nnnbr_, nnm2l_, nnp2l_, nnbr_, nm2l_, np2l_);
	k_p2m<<<blocks_for((long long)num_nodes_ * (p + 1), 256), 256, 0, stream_>>>(t, num_nodes_, p, sx_.ptr, sy_.ptr, sm_.ptr, mult_.ptr);
	const int per = fmm_nodes_per_block(p);
	for (int lev = levels_ - 1; lev >= 0; lev--)
	{
		const int c0 = level_start_[lev + 1], c1 = level_start_[lev + 2];
		k_m2m<<<blocks_for(c1 - c0, per), FMM_THREADS, 0, stream_>>>(t, c0, c1, p, binom_.ptr, mult_.ptr);
	}
	MLENS_HIP_CHECK(hipGetLastError());
	// M2L: FP64 recurrences inside k_local, or batched GEMMs on MFMA after it
	const bool mfma = m2l_mode_ != M2L_DIRECT;
	const bool f32 = m2l_mode_ == M2L_MFMA_F32 || (m2l_mode_ == M2L_MFMA && p <= 20);
	if (mfma)
	{
		m2l_prepare(p, f32);
		if (m2l_count_.count < 2) m2l_count_.alloc(2);
		MLENS_HIP_CHECK(hipMemsetAsync(m2l_count_.ptr, 0, 2 * sizeof(unsigned long long), stream_));
		if (!m2l_ev0_) MLENS_HIP_CHECK(hipEventCreate(&m2l_ev0_));
		if (!m2l_ev1_) MLENS_HIP_CHECK(hipEventCreate(&m2l_ev1_));
		MLENS_HIP_CHECK(hipEventRecord(m2l_ev0_, stream_));
		if (levels_ >= 2) m2l_all(p, f32);
		MLENS_HIP_CHECK(hipEventRecord(m2l_ev1_, stream_));
	}
	for (int lev = 2; lev <= levels_; lev++)
	{
		int l0 = level_start_[lev], l1 = level_start_[lev + 1];
		k_local<<<blocks_for(l1 - l0, per), FMM_THREADS, 0, stream_>>>(t, l0, l1, p, binom_.ptr, mult_.ptr, local_.ptr, sx_.ptr,
			sy_.ptr, sm_.ptr, mfma ? 0 : 1);
		MLENS_HIP_CHECK(hipGetLastError());
	}
	build_leaf_tables(lens);
	MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
	m2l_ms_ = 0;
	m2l_pairs_ = 0;
	m2l_f32_ = mfma && f32;
	if (mfma)
	{
		float ms = 0;
		MLENS_HIP_CHECK(hipEventElapsedTime(&ms, m2l_ev0_, m2l_ev1_));
		m2l_ms_ = ms;
		unsigned long long h[2];
		MLENS_HIP_CHECK(hipMemcpy(h, m2l_count_.ptr, sizeof(h), hipMemcpyDeviceToHost));
		m2l_pairs_ = (long long)h[0];
		if (h[1] & 1) throw HipError("an M2L source is not at one of the 40 offsets of its target's level", __FILE__, __LINE__);
	}
}

void Engine::build_leaf_tables(const LensParams& lens)
{
	const int nn = num_nodes_;
	const int SD = poly_stride_d(p_), SF = poly_stride_f(p_);
	leaf_geom_.alloc(size_t(num_leaves_) * 4);
	leaf_near_n_.alloc(num_leaves_);
	leaf_near_true_.alloc(num_leaves_);
	leaf_near_d_.alloc(size_t(num_leaves_) * MAX_NUM_STARS_DIRECT * 3);
	leaf_near_f_.alloc(size_t(num_leaves_) * MAX_NUM_STARS_DIRECT * 4);
	leaf_poly_d_.alloc(size_t(std::max(num_leaves_, 1)) * SD * 2);
	leaf_poly_f_.alloc(size_t(std::max(num_leaves_, 1)) * std::max(SF, 1) * 2);
	TreeView t = view(ncx_, ncy_, nhl_, nlevel_, nparent_, nchild0_, nbegin_, ncount_, nnnbr_, nnm2l_, nnp2l_, nnbr_, nm2l_, np2l_);
	k_leaf_tables<<<blocks_for(nn, 8), 256, 0, stream_>>>(t, nn, level_start_[levels_], last_level_leaf0_, p_, lens.theta * lens.theta, sx_.ptr, sy_.ptr,
		sm_.ptr, local_.ptr, leaf_of_node_.ptr, leaf_geom_.ptr, leaf_near_n_.ptr, leaf_near_true_.ptr, leaf_near_d_.ptr,
		leaf_near_f_.ptr,
		leaf_poly_d_.ptr, leaf_poly_f_.ptr);
	MLENS_HIP_CHECK(hipGetLastError());
}

void Engine::export_coeffs(int which, double* out) const
{
	const DeviceBuffer<double>& b = which ? local_ : mult_;
	MLENS_HIP_CHECK(hipMemcpy(out, b.ptr, size_t(num_nodes_) * (p_ + 1) * 2 * sizeof(double), hipMemcpyDeviceToHost));
}

}  // namespace mlens
