// Critical curves and caustics of a star field (ccf_functions.cuh, ccf.cuh).
//
// For every phase phi the critical curve points are the roots of
//   f(z, phi) = gamma - conj(d alpha / d zbar) - (1 - kappa - d alpha_smooth / dz) e^{-i phi},
// a rational function with a double pole at every star. All roots of one phi
// are refined together by Aberth's method (each Newton step corrected by the
// poles and by the other roots), starting at the centre phase of each branch
// from positions next to the stars, then stepping phi outwards in both
// directions with the previous phase's roots as starting points.
//
// On this GPU a wave of 64 lanes updates one root: the sums over all roots and
// all stars are split over its lanes, so a root update costs
// O((roots + stars) / 64) arithmetic per lane. Updates are simultaneous
// (Jacobi): an iteration reads one copy of the roots and writes the other, so
// the result does not depend on the order in which blocks run. Each branch and
// side is a chain of steps and iterations that only its own roots link; the
// blocks of a chain stay resident and meet at a barrier after each iteration,
// and leave a step as soon as every root has converged. Fields of more than
// 1024 stars, and a busy device, take a launch per iteration.
#include "shoot_common.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace mlens
{

namespace
{

constexpr double CCF_PI = 3.14159265358979323846;

// the derivative terms of the lens equation at z, in the node z falls in
struct CCTerms
{
	dcx S1, S2;     // sum over the node's near stars of m / (z - z_i)^2 and m / (z - z_i)^3
	dcx L1, L2;     // theta^2 / h^2 sum i(i-1) c_i dz^(i-2) and theta^2 / h^3 sum i(i-1)(i-2) c_i dz^(i-3)
	double ddz;     // d alpha_smooth / dz (real)
	dcx ddzb, d2s;  // d alpha_smooth / dzbar, d^2 alpha_smooth / dzbar^2
};

// alpha_star.cuh:55-114, alpha_local.cuh:52-108, alpha_smooth.cuh:142-316. With part < parts, only
// the near stars whose position in the node's near list is part (mod parts) enter S1 and S2, and the
// expansion and smooth terms are evaluated by part 0 only (zero elsewhere): the caller adds the parts.
template <bool LIN = false>
__device__ CCTerms cc_terms(const ShootArgs& a, int node, dcx z, bool second, int part = 0, int parts = 1)
{
	CCTerms t;
	double s1x = 0, s1y = 0, s2x = 0, s2y = 0;
	int seen = 0;
	auto range = [&](int b, int n) {
		// the first star of this range that belongs to this part
		const int first = ((part - seen) % parts + parts) % parts;
		seen += n;
		for (int s = b + first; s < b + n; s += parts)
		{
			const double dx = z.re - a.sx[s], dy = z.im - a.sy[s], m = a.sm[s];
			// 1 / (z - z_i) = conj(d) / |d|^2
			const double ir2 = dev::rcp64(dx * dx + dy * dy);
			const double ux = dx * ir2, uy = -dy * ir2;
			const double u2x = ux * ux - uy * uy, u2y = 2 * ux * uy;
			s1x += m * u2x;
			s1y += m * u2y;
			if (second)
			{
				s2x += m * (u2x * ux - u2y * uy);
				s2y += m * (u2x * uy + u2y * ux);
			}
		}
	};
	range(a.nbegin[node], a.ncount[node]);
	for (int j = 0; j < a.nnnbr[node]; j++)
	{
		const int nb = a.nnbr[8 * node + j];
		range(a.nbegin[nb], a.ncount[nb]);
	}
	t.S1 = dcx{s1x, s1y};
	t.S2 = dcx{s2x, s2y};
	t.L1 = t.L2 = t.ddzb = t.d2s = dcx{0, 0};
	t.ddz = 0;
	if (part != 0) return t;
	const double h = a.nhl[node];
	const dcx dz = dcx{(z.re - a.ncx[node]) / h, (z.im - a.ncy[node]) / h};
	const double* c = a.local + 2 * (long long)node * (a.p + 1);
	dcx l1 = {0, 0}, l2 = {0, 0};
	for (int i = a.p; i >= 2; i--)
	{
		l1 = dev::add(dev::mul(l1, dz), dev::scale(dcx{c[2 * i], c[2 * i + 1]}, double(i) * (i - 1)));
		if (second && i >= 3) l2 = dev::add(dev::mul(l2, dz), dev::scale(dcx{c[2 * i], c[2 * i + 1]}, double(i) * (i - 1) * (i - 2)));
	}
	t.L1 = dev::scale(l1, a.theta2 / (h * h));
	t.L2 = dev::scale(l2, a.theta2 / (h * h * h));
	if (LIN)
	{
		t.ddz = -a.kappastar;
		return t;
	}
	const dcx corner = dcx{a.corner_re, a.corner_im};
	dev::d_alpha_smooth(z, a.kappastar, a.rectangular, a.approx, a.taylor_smooth, corner, t.ddz, t.ddzb);
	t.d2s = second ? dev::d2_alpha_smooth(z, a.kappastar, a.rectangular, a.approx, a.taylor_smooth, corner) : dcx{0, 0};
	return t;
}

// f(z, phi) of ccf_functions.cuh:64-80 from the terms
__device__ __forceinline__ dcx cc_f0(const ShootArgs& a, const CCTerms& t, double phi)
{
	const double dwdz = (1 - a.kappa) - t.ddz;
	double sn, cs;
	sincos(phi, &sn, &cs);
	return dcx{a.gamma + a.theta2 * t.S1.re - t.L1.re - t.ddzb.re - dwdz * cs,
		a.theta2 * t.S1.im - t.L1.im + t.ddzb.im + dwdz * sn};
}

// largest possible error in 1/mu at a root (ccf_functions.cuh:204-211, 466-472)
__device__ __forceinline__ double cc_inv_mu_error(const ShootArgs& a, const CCTerms& t, dcx f0)
{
	const double af = dev::cabs(f0), dwdz = (1 - a.kappa) - t.ddz;
	return fmax(fabs(af * (af + 2 * dwdz)), fabs(af * (af - 2 * dwdz)));
}

// row r of the root array: its branch, its step from the branch centre and its phase
struct CCRow
{
	int row;
	double phi;
};

__device__ __forceinline__ CCRow cc_row(int c, int sgn, int j, int nphi, int nb)
{
	const int J = nphi / (2 * nb);
	CCRow r;
	r.row = c * (2 * J + 1) + J + sgn * j;
	r.phi = CCF_PI / nb + c * 2 * CCF_PI / nb + sgn * j * (2 * CCF_PI / nphi);
	return r;
}

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
	return v;
}

/*
The derivative terms of cc_terms at z in leaf `node` (the same in every lane), with one near star per lane,
S1 and S2 summed over the wave. Each lane fetches one near star (the leaf's table pads the list with massless
ones) and one coefficient of the expansion at the start, so that nothing below waits for memory.
*/
struct CCLeaf
{
	double x, y, m;     // this lane's near star
	double cre, cim;    // coefficient `lane` of the local expansion
	double cx, cy, h;
	int near;           // near stars in the table
};

__device__ __forceinline__ CCLeaf cc_load_leaf(const ShootArgs& a, int node)
{
	const int lane = threadIdx.x & 63;
	const long long L = a.leaf_of_node[node];
	CCLeaf f;
	f.near = a.leaf_near_n[L] & 0xffff;
	const double* s = a.near_d + (L * MAX_NUM_STARS_DIRECT + min(lane, MAX_NUM_STARS_DIRECT - 1)) * 3;
	f.x = s[0];
	f.y = s[1];
	f.m = s[2];
	const double* c = a.local + 2 * ((long long)node * (a.p + 1) + min(lane, a.p));
	f.cre = c[0];
	f.cim = c[1];
	f.cx = a.ncx[node];
	f.cy = a.ncy[node];
	f.h = a.nhl[node];
	return f;
}

__device__ __forceinline__ double lane_value(double v, int lane)
{
	const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
	const unsigned lo = __builtin_amdgcn_readlane(unsigned(b), lane), hi = __builtin_amdgcn_readlane(unsigned(b >> 32), lane);
	return __builtin_bit_cast(double, (static_cast<unsigned long long>(hi) << 32) | lo);
}

template <bool LIN>
__device__ __forceinline__ CCTerms cc_terms_leaf(const ShootArgs& a, const CCLeaf& f, dcx z)
{
	CCTerms t;
	t.S1 = t.S2 = dcx{0, 0};
	if (int(threadIdx.x & 63) < f.near)
	{
		const double dx = z.re - f.x, dy = z.im - f.y;
		const double ir2 = dev::rcp64(dx * dx + dy * dy);
		const double ux = dx * ir2, uy = -dy * ir2;
		const double u2x = ux * ux - uy * uy, u2y = 2 * ux * uy;
		t.S1.re += f.m * u2x;
		t.S1.im += f.m * u2y;
		t.S2.re += f.m * (u2x * ux - u2y * uy);
		t.S2.im += f.m * (u2x * uy + u2y * ux);
	}
	const dcx dz = dcx{(z.re - f.cx) / f.h, (z.im - f.cy) / f.h};
	dcx l1 = {0, 0}, l2 = {0, 0};
	for (int i = a.p; i >= 2; i--)
	{
		const dcx c = dcx{lane_value(f.cre, i), lane_value(f.cim, i)};
		l1 = dev::add(dev::mul(l1, dz), dev::scale(c, double(i) * (i - 1)));
		if (i >= 3) l2 = dev::add(dev::mul(l2, dz), dev::scale(c, double(i) * (i - 1) * (i - 2)));
	}
	t.L1 = dev::scale(l1, a.theta2 / (f.h * f.h));
	t.L2 = dev::scale(l2, a.theta2 / (f.h * f.h * f.h));
	t.ddz = -a.kappastar;
	t.ddzb = t.d2s = dcx{0, 0};
	if (LIN) return t;
	const dcx corner = dcx{a.corner_re, a.corner_im};
	dev::d_alpha_smooth(z, a.kappastar, a.rectangular, a.approx, a.taylor_smooth, corner, t.ddz, t.ddzb);
	t.d2s = dev::d2_alpha_smooth(z, a.kappastar, a.rectangular, a.approx, a.taylor_smooth, corner);
	return t;
}

// Roots cross between the blocks of a chain through these: relaxed atomics of device scope, which the
// per-XCD L2 caches do not hold back, so that nothing else cached (tree, stars) has to be invalidated.
__device__ __forceinline__ double load_shared(const double* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void store_shared(double* p, double v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

/*
The barrier after iteration `slot` of a chain of `blocks` blocks: each adds one to the low half of the slot's word
and its count of unconverged roots to the high half. Returns the chain's total (final, and so the same in every
block, once all have arrived), or -1 if some block polled `polls` times in vain and set *failed: an iteration of
millions of roots can take longer than the others wait, and the caller then starts the chain again without waiting.
Every slot is used once and starts at zero.
*/
constexpr int CCF_THREADS = 512;
constexpr int CCF_FIT = 2048;   // roots and stars of a chain that a block holds in LDS (32 KB each)
constexpr long long CCF_MEET_TICKS = 500000;   // 5 ms of the 100 MHz clock

/*
Whether every block of the launch is on the device at once, which the barriers need: the last block to arrive
decides that they are, a block that has waited 5 ms that they are not (other work holds the device), and all blocks
follow the one decision. state: blocks arrived in the low half, the decision (1 go, 2 no) above; starts at zero.
*/
__device__ bool all_resident(unsigned long long* state)
{
	__shared__ int go;
	if (threadIdx.x == 0)
	{
		constexpr unsigned long long GO = 1ull << 32, NO = 2ull << 32;
		const unsigned long long all = (unsigned long long)gridDim.x * gridDim.y;
		const long long t0 = wall_clock64();
		unsigned long long v = __hip_atomic_fetch_add(state, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
		for (;;)
		{
			if (v >> 32) break;
			const bool here = v == all, late = wall_clock64() - t0 > CCF_MEET_TICKS;
			if (here || late)
			{
				// decides unless the word has changed meanwhile; v is then its new value
				const unsigned long long want = v | (here ? GO : NO);
				if (__hip_atomic_compare_exchange_strong(state, &v, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
					v = want;
				continue;
			}
			__builtin_amdgcn_s_sleep(1);
			v = __hip_atomic_load(state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		}
		go = (v >> 32) == 1;
	}
	__syncthreads();
	return go;
}

__device__ int chain_barrier(unsigned long long* slot, int blocks, int active, int* failed, int polls)
{
	__shared__ int result;
	// this wave's stores have reached the coherence point; then every wave's have
	asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
	__syncthreads();
	if (threadIdx.x == 0)
	{
		unsigned long long v = __hip_atomic_fetch_add(slot, 1ull + ((unsigned long long)active << 32), __ATOMIC_RELAXED,
			__HIP_MEMORY_SCOPE_AGENT);
		int polled = 0;
		result = 0;
		do
		{
			v = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			if (int(v & 0xffffffffu) == blocks) break;
			if (polled++ >= polls || __hip_atomic_load(failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
			{
				__hip_atomic_store(failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				result = -1;
				break;
			}
			__builtin_amdgcn_s_sleep(1);
		} while (true);
		if (result == 0) result = int(v >> 32);
	}
	__syncthreads();
	const int r = result;
	asm volatile("" ::: "memory");
	return r;
}

/*
What an update of the root at z needs beside the sums over roots and stars: its leaf, from the previous iteration
while the root stays strictly inside it (there the tree descent would end in the same leaf), else by a fresh descent.
*/
struct CCPlace
{
	int node;
	bool leaf;
	CCLeaf f;
};

__device__ __forceinline__ void cc_find_place(const ShootArgs& a, dcx z, int* cache, CCPlace& p)
{
	const int cached = __builtin_amdgcn_readfirstlane(*cache);
	bool inside = false;
	if (cached >= 0)
	{
		const double h = a.nhl[cached] * (1 - 1e-12);
		inside = fabs(z.re - a.ncx[cached]) < h && fabs(z.im - a.ncy[cached]) < h;
	}
	p.node = __builtin_amdgcn_readfirstlane(inside ? cached : find_node(a, z.re, z.im));
	p.leaf = a.nchild0[p.node] < 0;
	if (!inside && (threadIdx.x & 63) == 0) *cache = p.leaf ? p.node : -1;
	if (p.leaf) p.f = cc_load_leaf(a, p.node);
}

// this lane's share of the sum of 1 / (z - x_q) over points q < n of a tile, leaving out point `skip`
__device__ __forceinline__ void cc_pair_sum(const double* x, const double* y, int n, int skip, dcx z, double& re, double& im)
{
	for (int q = threadIdx.x & 63; q < n; q += 64)
	{
		if (q == skip) continue;
		const double dx = z.re - x[q], dy = z.im - y[q];
		const double ir2 = dev::rcp64(dx * dx + dy * dy);
		re += dx * ir2;
		im -= dy * ir2;
	}
}

// The Aberth update of z from its lanes' shares of the sums over the other roots (r) and the poles (p): the new root
// (in lane 0), and whether it is final.
template <bool LIN>
__device__ __forceinline__ dcx cc_update(const ShootArgs& a, const CCPlace& place, dcx z, dcx r, dcx p, double phi, int circle_pole, bool& fin)
{
	CCTerms t;
	if (place.leaf)
		t = cc_terms_leaf<LIN>(a, place.f, z);
	else
	{
		// outside the root box; the tree's pointers are read here only
		const ShootArgs* cold = reinterpret_cast<const ShootArgs*>((const void*)__builtin_amdgcn_kernarg_segment_ptr());
		asm volatile("" : "+s"(cold));
		t = cc_terms<LIN>(*cold, place.node, z, true, threadIdx.x & 63, 64);
	}
	r.re = wave_sum(r.re);
	r.im = wave_sum(r.im);
	p.re = wave_sum(p.re);
	p.im = wave_sum(p.im);
	t.S1.re = wave_sum(t.S1.re);
	t.S1.im = wave_sum(t.S1.im);
	t.S2.re = wave_sum(t.S2.re);
	t.S2.im = wave_sum(t.S2.im);
	dcx zn = z;
	if ((threadIdx.x & 63) == 0)
	{
		const dcx f0 = cc_f0(a, t, phi);
		// 1/mu below 1e-9 (both bounds of ccf_functions.cuh:207-211): the root stays
		fin = cc_inv_mu_error(a, t, f0) < 1e-9;
		if (!fin)
		{
			const dcx f1 = dcx{-2 * a.theta2 * t.S2.re - t.L2.re - t.d2s.re, -2 * a.theta2 * t.S2.im - t.L2.im + t.d2s.im};
			dcx psum = dcx{2 * p.re, 2 * p.im};
			if (circle_pole)
			{
				const dcx iz = dev::cdiv(dcx{1, 0}, z);
				psum = dev::add(psum, dev::scale(iz, 2));
			}
			const dcx den = dev::add(f1, dev::mul(f0, dcx{psum.re - r.re, psum.im - r.im}));
			zn = dev::sub(z, dev::cdiv(f0, den));
			fin = dev::cabs(dev::sub(zn, z)) / sqrt(a.theta2) < 1e-9;
		}
	}
	return zn;
}

/*
Steps j0 .. j1 of chains first_chain + [0, gridDim.y) (ccf_functions.cuh:171-240, 309-386): chain c * sides + b is
branch c, side b (side 0 steps phi down, side 1 up; at j = 0 there is one side). A step starts from the roots of
the one before it and runs at most `iters` Aberth iterations; once every root of the chain has converged the rest
would change nothing and is left out. Blocks of eight waves, a wave per root at a time, root by root round the
chain's gridDim.x blocks; each holds all roots and stars in LDS, at most CCF_FIT of either. 137 stars (274 roots,
100 phases): 1.8 ms, against 4.5 ms with one launch per iteration. A step takes about seven iterations of 5 us, most
of which is the round trip through the barrier and the shared roots. Blocks of 256 or 1024 threads took 1.74 and
2.37 ms. rows: (nphi + nb) rows of nroots roots, the result; work: two copies of each chain's roots; slots: one word
for the launch, then iters words per step of each chain, zeroed. The blocks meet first: if they are not all resident
at once, the launch does nothing and failed[1] says so. (A cooperative launch would promise that they are, but the
device grants those to one process at a time.) If a block waits in vain at a barrier, failed[0] says so and all
leave. The work then goes out through k_ccf_iterate, with no waiting.
*/
template <bool LIN>
__global__ __launch_bounds__(CCF_THREADS) void k_ccf_chain(ShootArgs a, dcx* __restrict__ rows, double* work, char* __restrict__ fin,
	int* __restrict__ leaf_cache, unsigned long long* slots, int* failed, int nroots, int nstars, int circle_pole, int j0, int j1,
	int nphi, int nb, int sides, int iters, int first_chain, int polls)
{
	__shared__ double rx_s[CCF_FIT], ry_s[CCF_FIT], px_s[CCF_FIT], py_s[CCF_FIT];
	__shared__ int active_s;
	if (!all_resident(slots + first_chain))
	{
		if (threadIdx.x == 0) __hip_atomic_store(failed + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		return;
	}
	const int chain = first_chain + blockIdx.y;
	const int c = chain / sides, b = chain % sides;
	const int sgn = (sides == 1 || b == 1) ? 1 : -1;
	const int lane = threadIdx.x & 63;
	const int wave = __builtin_amdgcn_readfirstlane(int(blockIdx.x) * (CCF_THREADS / 64) + int(threadIdx.x >> 6));
	const int waves = int(gridDim.x) * (CCF_THREADS / 64);
	double* cur = work + 4ll * chain * nroots;   // (re, im) of every root, twice
	double* nxt = cur + 2ll * nroots;
	for (int i = threadIdx.x; i < nstars; i += CCF_THREADS)
	{
		px_s[i] = a.sx[i];
		py_s[i] = a.sy[i];
	}
	unsigned long long* slot = slots + nb * sides + (long long)chain * (j1 - j0 + 1) * iters;
	char* done = fin + ((long long)c * 2 + b) * nroots;
	int* leaves = leaf_cache + ((long long)c * 2 + b) * nroots;
	for (int j = j0; j <= j1; j++)
	{
		const CCRow R = cc_row(c, sgn, j, nphi, nb);
		for (int k = wave; k < nroots; k += waves)
			if (lane == 0) done[k] = 0;
		for (int it = 0; it < iters; it++)
		{
			if (threadIdx.x == 0) active_s = 0;
			for (int i = threadIdx.x; i < nroots; i += CCF_THREADS)
			{
				rx_s[i] = load_shared(cur + 2 * i);
				ry_s[i] = load_shared(cur + 2 * i + 1);
			}
			__syncthreads();
			for (int k = wave; k < nroots; k += waves)
			{
				const dcx z = dcx{rx_s[k], ry_s[k]};
				dcx zn = z;
				bool fin_now = true;
				if (!done[k])
				{
					CCPlace place;
					cc_find_place(a, z, leaves + k, place);
					dcx r = {0, 0}, p = {0, 0};
					cc_pair_sum(rx_s, ry_s, nroots, k, z, r.re, r.im);
					cc_pair_sum(px_s, py_s, nstars, -1, z, p.re, p.im);
					zn = cc_update<LIN>(a, place, z, r, p, R.phi, circle_pole, fin_now);
				}
				if (lane == 0)
				{
					store_shared(nxt + 2 * k, zn.re);
					store_shared(nxt + 2 * k + 1, zn.im);
					if (fin_now)
						done[k] = 1;
					else
						atomicAdd(&active_s, 1);
				}
			}
			__syncthreads();
			const int left = chain_barrier(slot + (long long)(j - j0) * iters + it, int(gridDim.x), active_s, failed, polls);
			if (left < 0) return;
			double* t = cur;
			cur = nxt;
			nxt = t;
			if (left == 0) break;
		}
		for (int k = wave; k < nroots; k += waves)
			if (lane < 2) reinterpret_cast<double*>(rows + (long long)R.row * nroots + k)[lane] = load_shared(cur + 2 * k + lane);
	}
}

/*
One iteration of step j of chains first_chain + [0, gridDim.y) by itself: four roots a block, a wave each, the same
sums in the same order. flip: which working copy is current; first, last: of the step's iterations. A block whose
roots are final copies them and leaves, so the iterations after the last change cost a launch each. Seven waves per
SIMD (70 VGPRs), which the sums over many roots need: 20000 stars, two phases, take 59 ms in all, 118 ms where
resident blocks of eight waves, one to a CU, read the roots past the caches once for every root of a wave.
*/
constexpr int CCF_ROOTS = 4;
constexpr int CCF_TILE = 256;

template <bool LIN>
__global__ __launch_bounds__(64 * CCF_ROOTS) void k_ccf_iterate(ShootArgs a, dcx* __restrict__ rows, dcx* work, char* __restrict__ fin,
	int* __restrict__ leaf_cache, int nroots, int nstars, int circle_pole, int j, int nphi, int nb, int sides, int first_chain, int flip,
	int first, int last)
{
	__shared__ double x_s[CCF_TILE], y_s[CCF_TILE];
	const int chain = first_chain + blockIdx.y;
	const int c = chain / sides, b = chain % sides;
	const CCRow R = cc_row(c, (sides == 1 || b == 1) ? 1 : -1, j, nphi, nb);
	const int lane = threadIdx.x & 63, k = __builtin_amdgcn_readfirstlane(int(blockIdx.x) * CCF_ROOTS + int(threadIdx.x >> 6));
	const dcx* cur = work + (2ll * chain + flip) * nroots;
	dcx* nxt = work + (2ll * chain + (1 - flip)) * nroots;
	char* done = fin + ((long long)c * 2 + b) * nroots;
	int* leaves = leaf_cache + ((long long)c * 2 + b) * nroots;
	const bool mine = k < nroots, active = mine && (first || !done[k]);
	const dcx z = mine ? cur[k] : dcx{0, 0};
	dcx zn = z;
	if (__syncthreads_or(active))
	{
		CCPlace place;
		if (active) cc_find_place(a, z, leaves + k, place);
		dcx r = {0, 0}, p = {0, 0};
		for (int t0 = 0; t0 < nroots; t0 += CCF_TILE)
		{
			const int i = t0 + threadIdx.x;
			const dcx v = i < nroots ? cur[i] : dcx{0, 0};
			__syncthreads();
			x_s[threadIdx.x] = v.re;
			y_s[threadIdx.x] = v.im;
			__syncthreads();
			if (active) cc_pair_sum(x_s, y_s, min(CCF_TILE, nroots - t0), k - t0, z, r.re, r.im);
		}
		for (int t0 = 0; t0 < nstars; t0 += CCF_TILE)
		{
			const int i = t0 + threadIdx.x;
			const dcx v = i < nstars ? dcx{a.sx[i], a.sy[i]} : dcx{0, 0};
			__syncthreads();
			x_s[threadIdx.x] = v.re;
			y_s[threadIdx.x] = v.im;
			__syncthreads();
			if (active) cc_pair_sum(x_s, y_s, min(CCF_TILE, nstars - t0), -1, z, p.re, p.im);
		}
		if (active)
		{
			bool fin_now = false;
			zn = cc_update<LIN>(a, place, z, r, p, R.phi, circle_pole, fin_now);
			if (lane == 0) done[k] = fin_now;
		}
	}
	if (mine && lane == 0)
	{
		nxt[k] = zn;
		if (last) rows[(long long)R.row * nroots + k] = zn;
	}
}
static_assert(CCF_TILE == 64 * CCF_ROOTS, "a thread stages a point");

// the working copies of chains first_chain + [0, gridDim.y) from the rows their first step starts from (step j)
__global__ void k_ccf_start(const dcx* __restrict__ rows, dcx* work, int nroots, int j, int nphi, int nb, int sides, int first_chain)
{
	const int k = blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= nroots) return;
	const int chain = first_chain + blockIdx.y, c = chain / sides, b = chain % sides;
	const CCRow from = cc_row(c, (sides == 1 || b == 1) ? 1 : -1, j, nphi, nb);
	work[2ll * chain * nroots + k] = rows[(long long)from.row * nroots + k];
}

/*
Per root of every row: the error bound on 1/mu (ccf_functions.cuh:430-474),
the transposed critical curve point (root-major, as written), the caustic
point (the lens equation, 496-516) and the magnification length scale
(134-160). err_bits collects the largest error as the bit pattern of a
non-negative double; nan_flag is set by any non-finite error.
*/
__global__ void k_ccf_finish(ShootArgs a, const dcx* __restrict__ roots, int nroots, int nphi, int nb, dcx* __restrict__ ccs,
	dcx* __restrict__ caustics, double* __restrict__ mu_scales, unsigned long long* err_bits, int* nan_flag)
{
	const long long total = (long long)(nphi + nb) * nroots;
	const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= total) return;
	const int rowi = int(i / nroots), k = int(i % nroots);
	const int J = nphi / (2 * nb);
	const int c = rowi / (2 * J + 1), s = rowi % (2 * J + 1) - J;
	const double phi = CCF_PI / nb + c * 2 * CCF_PI / nb + s * (2 * CCF_PI / nphi);
	const dcx z = roots[i];
	const int node = find_node(a, z.re, z.im);
	const CCTerms t = cc_terms(a, node, z, mu_scales != nullptr);
	const double err = cc_inv_mu_error(a, t, cc_f0(a, t, phi));
	if (!isfinite(err))
		atomicExch(nan_flag, 1);
	else
		atomicMax(err_bits, (unsigned long long)__double_as_longlong(err));
	const long long o = (long long)k * (nphi + nb) + rowi;
	ccs[o] = z;
	if (caustics)
	{
		const Deflection d = deflect_node<false>(a, node, z.re, z.im);
		caustics[o] = dcx{d.wx, d.wy};
	}
	if (mu_scales)
	{
		// ccf_functions.cuh:134-160
		const double dwdz = (1 - a.kappa) - t.ddz;
		const dcx dwdzb = dcx{a.gamma + a.theta2 * t.S1.re - t.L1.re - t.ddzb.re, -a.theta2 * t.S1.im + t.L1.im - t.ddzb.im};
		const dcx d2 = dcx{-2 * a.theta2 * t.S2.re - t.L2.re - t.d2s.re, 2 * a.theta2 * t.S2.im + t.L2.im - t.d2s.im};
		const dcx cct = dev::mul(dev::mul(dcx{0, -2}, dev::conj(dwdzb)), d2);
		const dcx ct = dev::add(dev::scale(cct, dwdz), dev::mul(dwdzb, dev::conj(cct)));
		mu_scales[o] = 1 / (2 * dev::cabs(ct));
	}
}

}  // namespace

CCFResult Engine::ccf_solve(const LensParams& lens, const double* init_roots, int nroots, int nphi, int nb, bool circle_pole,
	double* ccs, double* caustics, double* mu_scales, int init_iters, int step_iters)
{
	if (nroots < 1 || nphi < 2 || nb < 1 || nphi % (2 * nb) != 0) throw HipError("invalid critical curve sizes", __FILE__, __LINE__);
	if (!nstars_ || !num_nodes_) throw HipError("the critical curve solver needs the tree and the FMM", __FILE__, __LINE__);
	GridParams g;
	std::memset(&g, 0, sizeof(g));
	g.num_pixels[0] = g.num_pixels[1] = 1;
	g.half_length_y[0] = g.half_length_y[1] = 1;
	ShootArgs a = ShootArgsBuilder::make(lens, g, false);
	MLENS_TREE_ARGS(a)
	const int J = nphi / (2 * nb);
	const long long nrows = nphi + nb, total = nrows * nroots;
	// complex arrays as (re, im) pairs of doubles
	DeviceBuffer<double> Ab, Bb, Cb, Wb, M;
	DeviceBuffer<char> fin;
	DeviceBuffer<int> leaf_cache;
	DeviceBuffer<unsigned long long> err, slots;
	DeviceBuffer<int> flags;   // a non-finite error; a barrier that timed out; blocks that did not meet
	Ab.alloc(2 * total);
	Bb.alloc(2 * 4 * (size_t)nb * nroots);
	Cb.alloc(2 * total);
	if (caustics) Wb.alloc(2 * total);
	if (mu_scales) M.alloc(total);
	struct
	{
		dcx* ptr;
	} A{reinterpret_cast<dcx*>(Ab.ptr)}, C{reinterpret_cast<dcx*>(Cb.ptr)}, W{reinterpret_cast<dcx*>(Wb.ptr)};
	fin.alloc(2 * (size_t)nb * nroots);
	leaf_cache.alloc(2 * (size_t)nb * nroots);
	err.alloc(1);
	flags.alloc(3);
	const size_t nslots = 2 * (size_t)nb + std::max((size_t)nb * init_iters, 2 * (size_t)nb * J * step_iters);
	slots.alloc(nslots);
	MLENS_HIP_CHECK(hipMemsetAsync(A.ptr, 0, total * sizeof(dcx), stream_));
	MLENS_HIP_CHECK(hipMemsetAsync(leaf_cache.ptr, 0xff, 2 * (size_t)nb * nroots * sizeof(int), stream_));   // -1: none
	MLENS_HIP_CHECK(hipMemsetAsync(err.ptr, 0, sizeof(unsigned long long), stream_));
	MLENS_HIP_CHECK(hipMemsetAsync(flags.ptr, 0, 3 * sizeof(int), stream_));
	// starting roots at the centre row of each branch
	auto upload_start = [&](int first, int branches) {
		for (int c = first; c < first + branches; c++)
			MLENS_HIP_CHECK(hipMemcpyAsync(A.ptr + (long long)(c * (2 * J + 1) + J) * nroots, init_roots + 2 * (long long)c * nroots,
				nroots * sizeof(dcx), hipMemcpyHostToDevice, stream_));
	};
	upload_start(0, nb);
	// Steps j0 .. j1 of every chain. The blocks of a chain wait for each other, so all blocks of a launch must be
	// resident: they share out evenly over the chains what the device holds, no more than a chain has roots for;
	// chains beyond that go into further launches.
	const void* kernel = a.smooth_linear ? (const void*)k_ccf_chain<true> : (const void*)k_ccf_chain<false>;
	int per_cu = 0;
	MLENS_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, CCF_THREADS, 0));
	const int resident = num_cus_ * std::max(1, per_cu);
	// resident chains for fields that fit a block's LDS: 20 stars 1.5 against 2.9 ms, 500 stars 3.6 against 5.0, 1000
	// stars 3.0 against 3.4; from there on the pair sums count, not the launches. Until a block has waited in vain.
	bool together = ccf_together_ && nroots <= CCF_FIT && nstars_ <= CCF_FIT;
	auto sweep = [&](int from, int j0, int j1, int sides, int iters) {
		if (j1 < j0 || iters < 1) return;
		const int chains = nb * sides, waves = CCF_THREADS / 64;
		const unsigned row_blocks = blocks_for(nroots, 256);
		dcx* work = reinterpret_cast<dcx*>(Bb.ptr);
		int* bad = flags.ptr + 1;
		const int ns = nstars_, pole = circle_pole ? 1 : 0;
		auto chain_steps = [&](int first, int here) {
			const int blocks = std::max(1, std::min((nroots + waves - 1) / waves, resident / here));
			auto kernel = a.smooth_linear ? k_ccf_chain<true> : k_ccf_chain<false>;
			kernel<<<dim3(unsigned(blocks), unsigned(here)), CCF_THREADS, 0, stream_>>>(a, A.ptr, Bb.ptr, fin.ptr, leaf_cache.ptr,
				slots.ptr, bad, nroots, ns, pole, j0, j1, nphi, nb, sides, iters, first, ccf_polls_);
			MLENS_HIP_CHECK(hipGetLastError());
		};
		auto iterations = [&](int first, int here) {
			auto kernel = a.smooth_linear ? k_ccf_iterate<true> : k_ccf_iterate<false>;
			const dim3 grid(unsigned((nroots + CCF_ROOTS - 1) / CCF_ROOTS), unsigned(here));
			for (int j = j0, n = 0; j <= j1; j++)
				for (int it = 0; it < iters; it++, n++)
					kernel<<<grid, 64 * CCF_ROOTS, 0, stream_>>>(a, A.ptr, work, fin.ptr, leaf_cache.ptr, nroots, ns, pole, j, nphi, nb,
						sides, first, n & 1, it == 0, it == iters - 1);
			MLENS_HIP_CHECK(hipGetLastError());
		};
		auto start = [&](int first, int here) {
			k_ccf_start<<<dim3(row_blocks, unsigned(here)), 256, 0, stream_>>>(A.ptr, work, nroots, from, nphi, nb, sides, first);
			MLENS_HIP_CHECK(hipGetLastError());
		};
		start(0, chains);
		MLENS_HIP_CHECK(hipMemsetAsync(slots.ptr, 0, (chains + (size_t)chains * (j1 - j0 + 1) * iters) * sizeof(unsigned long long), stream_));
		const int group = std::min(chains, resident);
		for (int first = 0; first < chains; first += group)
		{
			const int here = std::min(group, chains - first);
			int nf[2] = {0, 1};
			if (together)
			{
				MLENS_HIP_CHECK(hipMemsetAsync(bad, 0, sizeof(nf), stream_));
				chain_steps(first, here);
				MLENS_HIP_CHECK(hipMemcpyAsync(nf, bad, sizeof(nf), hipMemcpyDeviceToHost, stream_));
				MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
			}
			if (!nf[0] && !nf[1]) continue;
			if (nf[0])
			{
				// some blocks have gone on: again from where the chains started (the first sweep writes that row)
				together = false;
				if (j0 == from) upload_start(first, here);
				start(first, here);
			}
			iterations(first, here);
		}
	};
	CCFResult r;
	MLENS_HIP_CHECK(hipEventRecord(ev0_, stream_));
	sweep(0, 0, 0, 1, init_iters);
	MLENS_HIP_CHECK(hipEventRecord(ev1_, stream_));
	MLENS_HIP_CHECK(hipEventSynchronize(ev1_));
	float ms = 0;
	MLENS_HIP_CHECK(hipEventElapsedTime(&ms, ev0_, ev1_));
	r.t_init_ms = ms;
	MLENS_HIP_CHECK(hipEventRecord(ev0_, stream_));
	if (step_iters > 0) sweep(0, 1, J, 2, step_iters);
	MLENS_HIP_CHECK(hipEventRecord(ev1_, stream_));
	MLENS_HIP_CHECK(hipEventSynchronize(ev1_));
	MLENS_HIP_CHECK(hipEventElapsedTime(&ms, ev0_, ev1_));
	r.t_ccs_ms = ms;
	MLENS_HIP_CHECK(hipEventRecord(ev0_, stream_));
	k_ccf_finish<<<blocks_for(total, 256), 256, 0, stream_>>>(a, A.ptr, nroots, nphi, nb, C.ptr, caustics ? W.ptr : nullptr,
		mu_scales ? M.ptr : nullptr, err.ptr, flags.ptr);
	MLENS_HIP_CHECK(hipGetLastError());
	MLENS_HIP_CHECK(hipEventRecord(ev1_, stream_));
	MLENS_HIP_CHECK(hipEventSynchronize(ev1_));
	MLENS_HIP_CHECK(hipEventElapsedTime(&ms, ev0_, ev1_));
	r.t_caustics_ms = ms;
	unsigned long long eb = 0;
	int nf = 0;
	MLENS_HIP_CHECK(hipMemcpy(&eb, err.ptr, sizeof(eb), hipMemcpyDeviceToHost));
	MLENS_HIP_CHECK(hipMemcpy(&nf, flags.ptr, sizeof(nf), hipMemcpyDeviceToHost));
	std::memcpy(&r.max_error, &eb, sizeof(double));
	r.has_nan = nf != 0;
	MLENS_HIP_CHECK(hipMemcpy(ccs, C.ptr, total * sizeof(dcx), hipMemcpyDeviceToHost));
	if (caustics) MLENS_HIP_CHECK(hipMemcpy(caustics, W.ptr, total * sizeof(dcx), hipMemcpyDeviceToHost));
	if (mu_scales) MLENS_HIP_CHECK(hipMemcpy(mu_scales, M.ptr, total * sizeof(double), hipMemcpyDeviceToHost));
	return r;
}

}  // namespace mlens
