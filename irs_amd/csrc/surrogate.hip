// The histogram surrogate: a multilayer perceptron mapping lens parameters
// to the 128-bin log10 magnification histogram of a map, trained and run on
// the GPU by the kernels below.
//
// Network: 6 inputs (zero-padded to 16) -> 256 -> 256 -> 256 -> 128 logits,
// SiLU activations, softmax output, cross-entropy against the normalised
// histogram. Products run on the matrix cores in BF16 with FP32 accumulation
// (v_mfma_f32_16x16x16_bf16): every GEMM operand is stored in BF16, every
// result, pre-activation, gradient and the Adam state in FP32; the master
// weights are FP32 and their BF16 copies are refreshed after each step.
#include "surrogate.hpp"

#include "philox.hpp"

#include <cmath>
#include <cstring>
#include <vector>

namespace mlens
{

namespace
{

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (NaN kept quiet)
__host__ __device__ inline unsigned short to_bf16(float x)
{
	unsigned u;
	std::memcpy(&u, &x, 4);
	if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
	u += 0x7fffu + ((u >> 16) & 1u);
	return (unsigned short)(u >> 16);
}

__device__ inline float sigmoidf(float z) { return 1.0f / (1.0f + expf(-z)); }

/*
Products: one wave per 16 x 16 tile, C[m][n] = sum_k A(m, k) B(k, n) in steps of
16, k ascending. Lane l feeds A[l % 16][4 (l / 16) + j] and
B[4 (l / 16) + j][l % 16], j = 0..3, and holds C[4 (l / 16) + r][l % 16]. Every
operand is stored so that a lane's four values along k are consecutive: one
8-byte read each.
*/
__device__ __forceinline__ bf16x4 load4(const unsigned short* p) { return *reinterpret_cast<const bf16x4*>(p); }
__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }

__host__ __device__ constexpr int net_dim(int l) { return l == 0 ? SURR_PIN : (l == SURR_LAYERS ? SURR_NOUT : SURR_HIDDEN); }

// offsets of a layer's weights [out x in] and biases in the parameter vector
__host__ __device__ constexpr int net_w(int l)
{
	int off = 0;
	for (int i = 0; i < l; i++) off += net_dim(i + 1) * net_dim(i) + net_dim(i + 1);
	return off;
}
__host__ __device__ constexpr int net_b(int l) { return net_w(l) + net_dim(l + 1) * net_dim(l); }

/*
Sixteen rows of the batch through the whole network, one block each: wave w owns
column tile w of every layer, activations pass through LDS, and the next layer's
weights are fetched while the current one is computed. With TRAIN the block goes
on to the loss, G = (P - T) / M (T rows sum to one), and back through the layers,
each dZ = dH SiLU'(Z), SiLU'(z) = s (1 + z (1 - s)), s = sigmoid(z): a wave holds
the pre-activations of its tiles in the lanes that get their gradients. The pass
is bound by its chain of reads and barriers. A request of 16 rows takes 40 us in
all; with a launch per product and per activation (nine launches, 69 us of
kernels) it took 104 us. An epoch of 16 steps of 256 rows takes 1.8 ms in all,
against 7.5 ms with 35 launches and a wait for the loss per step.
w: FP32 parameters (biases); w16, wt16: BF16 weights [out x in] and [in x out].
*/
constexpr int NET_THREADS = 1024;
constexpr int NET_ROWS = 16;
constexpr int NET_LDA = SURR_HIDDEN + 8;   // row stride of the activations in LDS

template <bool TRAIN>
__global__ __launch_bounds__(NET_THREADS) void k_net(const float* __restrict__ w, const unsigned short* __restrict__ w16,
	const unsigned short* __restrict__ wt16, const unsigned short* __restrict__ X, const int* __restrict__ idx,
	const float* __restrict__ T, int rows, float* __restrict__ P, float* __restrict__ loss, float inv_m, NetTrace tr)
{
	__shared__ __align__(16) unsigned short act[2][NET_ROWS * NET_LDA];
	__shared__ __align__(16) float out[NET_ROWS][SURR_NOUT + 4];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int i = lane & 15, kq = lane >> 4;
	const int m0 = blockIdx.x * NET_ROWS;
	const int col = wave * 16 + i;
	constexpr int STEPS = SURR_HIDDEN / 16;
	bf16x4 wa[STEPS], wb[STEPS];
	f32x4 z[SURR_LAYERS - 1];
	// `steps` operands of a weight matrix with rows of `in`, from row `col` on
	auto fetch = [&](bf16x4* to, const unsigned short* from, int in, int steps) {
#pragma unroll
		for (int k = 0; k < STEPS; k++)
			if (k < steps) to[k] = load4(from + (long long)col * in + k * 16 + kq * 4);
	};
	auto product = [&](const unsigned short* a, const bf16x4* b, int steps) {
		f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
		for (int k = 0; k < STEPS; k++)
			if (k < steps) acc = mfma16(load4(a + i * NET_LDA + k * 16 + kq * 4), b[k], acc);
		return acc;
	};
	// four rows of column `col`, into LDS and, training, to the trace
	auto put = [&](unsigned short* lds, const unsigned short v[4], unsigned short* trace) {
#pragma unroll
		for (int r = 0; r < 4; r++) lds[(4 * kq + r) * NET_LDA + col] = v[r];
		if (TRAIN)
		{
			bf16x4 t;
#pragma unroll
			for (int r = 0; r < 4; r++) t[r] = (short)v[r];
			*reinterpret_cast<bf16x4*>(trace + (long long)col * tr.ld + m0 + 4 * kq) = t;
		}
	};
	fetch(wa, w16 + net_w(0), SURR_PIN, 1);
	fetch(wb, w16 + net_w(1), SURR_HIDDEN, STEPS);
	if (threadIdx.x < NET_ROWS * SURR_PIN)
	{
		const int r = threadIdx.x / SURR_PIN, c = threadIdx.x % SURR_PIN;
		const long long src = idx ? idx[m0 + r] : m0 + r;
		const unsigned short x = X[src * SURR_PIN + c];
		act[0][r * NET_LDA + c] = x;
		if (TRAIN) tr.in[0][(long long)c * tr.ld + m0 + r] = x;
	}
	__syncthreads();
	unsigned short *src = act[0], *dst = act[1];
	auto swap = [&]() {
		unsigned short* t = src;
		src = dst;
		dst = t;
	};
#pragma unroll
	for (int l = 0; l < SURR_LAYERS - 1; l++)
	{
		// the layer's weights are in wa (l even) or wb; the next one's are on their way
		z[l] = product(src, l % 2 ? wb : wa, net_dim(l) / 16);
		if (l == 0) fetch(wa, w16 + net_w(2), SURR_HIDDEN, STEPS);
		if (l == 1 && wave < SURR_NOUT / 16) fetch(wb, w16 + net_w(3), SURR_HIDDEN, STEPS);
		const float bias = w[net_b(l) + col];
		unsigned short h[4];
#pragma unroll
		for (int r = 0; r < 4; r++)
		{
			z[l][r] = z[l][r] + bias;
			h[r] = to_bf16(z[l][r] * sigmoidf(z[l][r]));
		}
		put(dst, h, TRAIN ? tr.in[l + 1] : nullptr);
		__syncthreads();
		swap();
	}
	if (wave < SURR_NOUT / 16)
	{
		const f32x4 y = product(src, wb, STEPS);
		const float bias = w[net_b(SURR_LAYERS - 1) + col];
#pragma unroll
		for (int r = 0; r < 4; r++) out[4 * kq + r][col] = y[r] + bias;
	}
	// the last layer's backward weights: rows of W^T
	if (TRAIN) fetch(wa, wt16 + net_w(3), SURR_NOUT, SURR_NOUT / 16);
	__syncthreads();
	{
		// one wave per row of 128 logits: softmax, and the loss -sum T log P with log p = z - mx - log s
		const int row = wave;
		const float z0 = out[row][lane], z1 = out[row][lane + 64];
		float mx = fmaxf(z0, z1);
		for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
		float e0 = expf(z0 - mx), e1 = expf(z1 - mx);
		float s = e0 + e1;
		for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
		const float ls = logf(s);
		const float p0 = e0 / s, p1 = e1 / s;
		if (!TRAIN)
		{
			if (m0 + row < rows)
			{
				P[(long long)(m0 + row) * SURR_NOUT + lane] = p0;
				P[(long long)(m0 + row) * SURR_NOUT + lane + 64] = p1;
			}
			return;
		}
		const float* t = T + (long long)idx[m0 + row] * SURR_NOUT;
		const float t0 = t[lane], t1 = t[lane + 64];
		float l = -(t0 * (z0 - mx - ls) + t1 * (z1 - mx - ls));
		for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
		if (lane == 0) loss[m0 + row] = l;
		const float g0 = (p0 - t0) * inv_m, g1 = (p1 - t1) * inv_m;
		out[row][lane] = g0;
		out[row][lane + 64] = g1;
		dst[row * NET_LDA + lane] = to_bf16(g0);
		dst[row * NET_LDA + lane + 64] = to_bf16(g1);
	}
	__syncthreads();
	swap();
	// the output gradient's trace
	for (int q = threadIdx.x; q < SURR_NOUT * NET_ROWS / 4; q += NET_THREADS)
	{
		const int n = q >> 2, r0 = (q & 3) * 4;
		float4 g;
		bf16x4 t;
#pragma unroll
		for (int r = 0; r < 4; r++)
		{
			(&g.x)[r] = out[r0 + r][n];
			t[r] = (short)src[(r0 + r) * NET_LDA + n];
		}
		*reinterpret_cast<float4*>(tr.dz32[SURR_LAYERS - 1] + (long long)n * tr.ld + m0 + r0) = g;
		*reinterpret_cast<bf16x4*>(tr.dz16[SURR_LAYERS - 1] + (long long)n * tr.ld + m0 + r0) = t;
	}
	// dH of layer l - 1 = dZ_l W_l, then dZ of it
#pragma unroll
	for (int l = SURR_LAYERS - 1; l >= 1; l--)
	{
		const bool even = (SURR_LAYERS - 1 - l) % 2 == 0;
		if (l > 1) fetch(even ? wb : wa, wt16 + net_w(l - 1), net_dim(l), net_dim(l) / 16);
		const f32x4 dh = product(src, even ? wa : wb, net_dim(l + 1) / 16);
		float4 d;
		unsigned short d16[4];
#pragma unroll
		for (int r = 0; r < 4; r++)
		{
			const float zz = z[l - 1][r], sg = sigmoidf(zz);
			(&d.x)[r] = dh[r] * (sg * (1.0f + zz * (1.0f - sg)));
			d16[r] = to_bf16((&d.x)[r]);
		}
		*reinterpret_cast<float4*>(tr.dz32[l - 1] + (long long)col * tr.ld + m0 + 4 * kq) = d;
		put(dst, d16, tr.dz16[l - 1]);
		__syncthreads();
		swap();
	}
}

/*
Parameter gradients from the trace, and with ADAM the step of Adam with decoupled
weight decay (Loshchilov & Hutter 2019) on the FP32 master weights where they
come out, refreshing both BF16 copies; without it they go to g. A wave per 16 x 16 tile of
dW_l = dZ_l^T H_(l-1), the batch's rows ascending; the blocks after the tiles take
the biases, db[n] = sum_m dZ[m][n], a thread each (decay 0). Launched apart, the bias sums alone,
one thread walking a column of dZ, took 53 us a layer.
*/
struct AdamArgs
{
	float *w, *m, *v;
	unsigned short *w16, *wt16;
	float lr, b1, b2, eps, c1, c2, wd;
};

__device__ __forceinline__ float adam_step(const AdamArgs& a, long long i, float gi, float wd)
{
	const float mi = a.b1 * a.m[i] + (1.0f - a.b1) * gi;
	const float vi = a.b2 * a.v[i] + (1.0f - a.b2) * gi * gi;
	a.m[i] = mi;
	a.v[i] = vi;
	float wi = a.w[i] * (1.0f - a.lr * wd);
	wi -= a.lr * (mi * a.c1) / (sqrtf(vi * a.c2) + a.eps);
	a.w[i] = wi;
	return wi;
}

constexpr int GRAD_WAVES = 4;
constexpr int net_tiles(int l) { return net_dim(l + 1) / 16 * (net_dim(l) / 16); }
constexpr int GRAD_TILES = net_tiles(0) + net_tiles(1) + net_tiles(2) + net_tiles(3);
constexpr int GRAD_BIASES = 3 * SURR_HIDDEN + SURR_NOUT;
static_assert(SURR_LAYERS == 4 && GRAD_TILES % GRAD_WAVES == 0, "tile blocks are full");
constexpr int GRAD_TILE_BLOCKS = GRAD_TILES / GRAD_WAVES;
constexpr int GRAD_BLOCKS = GRAD_TILE_BLOCKS + (GRAD_BIASES + 64 * GRAD_WAVES - 1) / (64 * GRAD_WAVES);

template <bool ADAM>
__global__ __launch_bounds__(64 * GRAD_WAVES) void k_net_gradients(NetTrace tr, AdamArgs a, float* __restrict__ g)
{
	const int M = tr.ld;
	if (blockIdx.x >= GRAD_TILE_BLOCKS)
	{
		int n = int(blockIdx.x - GRAD_TILE_BLOCKS) * 64 * GRAD_WAVES + threadIdx.x;
		if (n >= GRAD_BIASES) return;
		const int l = min(n / SURR_HIDDEN, SURR_LAYERS - 1);
		n -= l * SURR_HIDDEN;
		const float4* d = reinterpret_cast<const float4*>(tr.dz32[l] + (long long)n * M);
		float s = 0.0f;
#pragma unroll 4
		for (int m = 0; m < M / 4; m++)
		{
			const float4 v = d[m];
			s += v.x;
			s += v.y;
			s += v.z;
			s += v.w;
		}
		if (ADAM)
			adam_step(a, net_b(l) + n, s, 0.0f);
		else
			g[net_b(l) + n] = s;
		return;
	}
	int tile = blockIdx.x * GRAD_WAVES + (threadIdx.x >> 6), l = 0;
	while (tile >= net_tiles(l)) tile -= net_tiles(l++);
	const int K = net_dim(l), N = net_dim(l + 1);
	const int tn = tile / (K / 16), tk = tile - tn * (K / 16);
	const int lane = threadIdx.x & 63, i = lane & 15, kq = lane >> 4;
	const unsigned short* d = tr.dz16[l] + (long long)(tn * 16 + i) * M + kq * 4;
	const unsigned short* h = tr.in[l] + (long long)(tk * 16 + i) * M + kq * 4;
	f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
	for (int m = 0; m < M; m += 16) acc = mfma16(load4(d + m), load4(h + m), acc);
	const int k = tk * 16 + i, n0 = tn * 16 + kq * 4;
	bf16x4 t;
#pragma unroll
	for (int r = 0; r < 4; r++)
	{
		const long long at = net_w(l) + (long long)(n0 + r) * K + k;
		if (ADAM)
		{
			const unsigned short b = to_bf16(adam_step(a, at, acc[r], a.wd));
			a.w16[at] = b;
			t[r] = (short)b;
		}
		else
			g[at] = acc[r];
	}
	if (ADAM) *reinterpret_cast<bf16x4*>(a.wt16 + net_w(l) + (long long)k * N + n0) = t;
}

// the BF16 copies of the weights, [out x in] and [in x out]
__global__ void k_net_copies(const float* __restrict__ w, unsigned short* __restrict__ w16, unsigned short* __restrict__ wt16)
{
	const int l = blockIdx.y, K = net_dim(l), N = net_dim(l + 1);
	const int g = blockIdx.x * blockDim.x + threadIdx.x;
	if (g >= N * K) return;
	const unsigned short b = to_bf16(w[net_w(l) + g]);
	w16[net_w(l) + g] = b;
	wt16[net_w(l) + (g % K) * N + g / K] = b;
}

inline unsigned blocks(long long n, int t) { return unsigned((n + t - 1) / t); }

}  // namespace

Surrogate::Surrogate(int max_batch, uint32_t seed) : max_batch_((max_batch + 15) / 16 * 16)
{
	MLENS_HIP_CHECK(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
	// parameter layout: W_l [out x in] then b_l [out] for l = 0..3
	nparams_ = net_w(SURR_LAYERS);
	w_.alloc(nparams_);
	g_.alloc(nparams_);
	m_.alloc(nparams_);
	v_.alloc(nparams_);
	w16_.alloc(nparams_);
	wt16_.alloc(nparams_);
	// He-uniform weights from Philox (key = seed), zero biases; padded input columns stay zero
	std::vector<float> w(nparams_, 0.0f);
	for (int l = 0; l < SURR_LAYERS; l++)
	{
		const int fin = l == 0 ? SURR_NIN : net_dim(l);
		const float a = std::sqrt(6.0f / float(fin));
		for (int o = 0; o < net_dim(l + 1); o++)
			for (int i = 0; i < fin; i++)
			{
				const uint64_t k = net_w(l) + size_t(o) * net_dim(l) + i;
				uint32_t ctr[4] = {uint32_t(k), uint32_t(k >> 32), 7u, 0u}, key[2] = {seed, 0x5eed5eedu}, r[4];
				philox4x32_10(ctr, key, r);
				const float u = float(r[0] >> 8) * (1.0f / 16777216.0f);
				w[k] = a * (2.0f * u - 1.0f);
			}
	}
	set_params(w.data());
}

Surrogate::~Surrogate()
{
	if (stream_)
	{
		(void)hipStreamSynchronize(stream_);
		(void)hipStreamDestroy(stream_);
	}
	if (small_) (void)hipHostFree(small_);
}

void Surrogate::set_params(const float* host)
{
	MLENS_HIP_CHECK(hipMemcpy(w_.ptr, host, nparams_ * sizeof(float), hipMemcpyHostToDevice));
	k_net_copies<<<dim3(blocks(SURR_HIDDEN * SURR_HIDDEN, 256), SURR_LAYERS), 256, 0, stream_>>>(w_.ptr, w16_.ptr, wt16_.ptr);
	MLENS_HIP_CHECK(hipGetLastError());
	MLENS_HIP_CHECK(hipMemsetAsync(m_.ptr, 0, nparams_ * sizeof(float), stream_));
	MLENS_HIP_CHECK(hipMemsetAsync(v_.ptr, 0, nparams_ * sizeof(float), stream_));
	MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
	step_ = 0;
}

void Surrogate::get_params(float* host) const
{
	MLENS_HIP_CHECK(hipMemcpy(host, w_.ptr, nparams_ * sizeof(float), hipMemcpyDeviceToHost));
}

// the trace of a training pass over M rows
NetTrace Surrogate::trace(int M)
{
	size_t n16 = 0, n32 = 0;
	for (int l = 0; l < SURR_LAYERS; l++)
	{
		n16 += net_dim(l) + net_dim(l + 1);
		n32 += net_dim(l + 1);
	}
	trace16_.alloc(n16 * max_batch_);
	trace32_.alloc(n32 * max_batch_);
	NetTrace t;
	unsigned short* p = trace16_.ptr;
	float* q = trace32_.ptr;
	for (int l = 0; l < SURR_LAYERS; l++)
	{
		t.in[l] = p;
		p += (size_t)net_dim(l) * M;
		t.dz16[l] = p;
		p += (size_t)net_dim(l + 1) * M;
		t.dz32[l] = q;
		q += (size_t)net_dim(l + 1) * M;
	}
	t.ld = M;
	return t;
}

static double mean_loss(const float* loss, int M)
{
	double s = 0;
	for (int r = 0; r < M; r++) s += loss[r];
	return s / M;
}

void Surrogate::load_data(const float* x, const float* t, int n)
{
	// inputs padded to SURR_PIN columns and stored in BF16; targets FP32
	std::vector<unsigned short> xp(size_t(n) * SURR_PIN, 0);
	for (int r = 0; r < n; r++)
		for (int c = 0; c < SURR_NIN; c++) xp[size_t(r) * SURR_PIN + c] = to_bf16(x[size_t(r) * SURR_NIN + c]);
	xall_.alloc(xp.size());
	tall_.alloc(size_t(n) * SURR_NOUT);
	MLENS_HIP_CHECK(hipMemcpyAsync(xall_.ptr, xp.data(), xp.size() * sizeof(unsigned short), hipMemcpyHostToDevice, stream_));
	MLENS_HIP_CHECK(hipMemcpyAsync(tall_.ptr, t, size_t(n) * SURR_NOUT * sizeof(float), hipMemcpyHostToDevice, stream_));
	MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
	ndata_ = n;
}

/* `steps` Adam steps, step k on rows[k M .. (k + 1) M) of the loaded set at rate lr[k]; the mean loss of each.
   Two launches a step and one wait in all: the losses stay on the device until the last step. */
void Surrogate::train(const int* rows, int steps, int M, const float* lr, float wd, double* losses)
{
	if (M <= 0 || M > max_batch_ || M % 16) throw HipError("surrogate batch must be a positive multiple of 16 within the maximum", __FILE__, __LINE__);
	if (steps < 0) throw HipError("a surrogate cannot train a negative number of steps", __FILE__, __LINE__);
	const size_t total = size_t(steps) * M;
	for (size_t r = 0; r < total; r++)
		if (rows[r] < 0 || rows[r] >= ndata_) throw HipError("surrogate row index outside the training set", __FILE__, __LINE__);
	if (total == 0) return;
	idx_.alloc(total);
	loss_.alloc(total);
	const NetTrace tr = trace(M);
	MLENS_HIP_CHECK(hipMemcpyAsync(idx_.ptr, rows, total * sizeof(int), hipMemcpyHostToDevice, stream_));
	for (int k = 0; k < steps; k++)
	{
		k_net<true><<<M / NET_ROWS, NET_THREADS, 0, stream_>>>(w_.ptr, w16_.ptr, wt16_.ptr, xall_.ptr, idx_.ptr + size_t(k) * M, tall_.ptr,
			M, nullptr, loss_.ptr + size_t(k) * M, 1.0f / float(M), tr);
		step_++;
		const float b1 = 0.9f, b2 = 0.999f;
		const float c1 = 1.0f / (1.0f - std::pow(b1, float(step_))), c2 = 1.0f / (1.0f - std::pow(b2, float(step_)));
		// the zero-padded input columns of W_0 get zero gradients and stay zero
		const AdamArgs a{w_.ptr, m_.ptr, v_.ptr, w16_.ptr, wt16_.ptr, lr[k], b1, b2, 1e-8f, c1, c2, wd};
		k_net_gradients<true><<<GRAD_BLOCKS, 64 * GRAD_WAVES, 0, stream_>>>(tr, a, nullptr);
		MLENS_HIP_CHECK(hipGetLastError());
	}
	std::vector<float> loss(total);
	MLENS_HIP_CHECK(hipMemcpyAsync(loss.data(), loss_.ptr, total * sizeof(float), hipMemcpyDeviceToHost, stream_));
	MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
	for (int k = 0; k < steps; k++) losses[k] = mean_loss(loss.data() + size_t(k) * M, M);
}

double Surrogate::train_step(const int* rows, int M, float lr, float wd)
{
	double loss = 0;
	train(rows, 1, M, &lr, wd, &loss);
	return loss;
}

double Surrogate::gradients(const float* x, const float* t, int n, float* grads)
{
	std::vector<int> rows(n);
	for (int i = 0; i < n; i++) rows[i] = i;
	load_data(x, t, n);
	if (n <= 0 || n % 16) throw HipError("gradient batch must be a multiple of 16", __FILE__, __LINE__);
	if (n > max_batch_) throw HipError("gradient batch must be within the surrogate's maximum", __FILE__, __LINE__);
	idx_.alloc(n);
	loss_.alloc(n);
	const NetTrace tr = trace(n);
	MLENS_HIP_CHECK(hipMemcpyAsync(idx_.ptr, rows.data(), n * sizeof(int), hipMemcpyHostToDevice, stream_));
	k_net<true><<<n / NET_ROWS, NET_THREADS, 0, stream_>>>(w_.ptr, w16_.ptr, wt16_.ptr, xall_.ptr, idx_.ptr, tall_.ptr, n, nullptr,
		loss_.ptr, 1.0f / float(n), tr);
	k_net_gradients<false><<<GRAD_BLOCKS, 64 * GRAD_WAVES, 0, stream_>>>(tr, AdamArgs{}, g_.ptr);
	MLENS_HIP_CHECK(hipGetLastError());
	std::vector<float> loss(n);
	MLENS_HIP_CHECK(hipMemcpyAsync(loss.data(), loss_.ptr, n * sizeof(float), hipMemcpyDeviceToHost, stream_));
	MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
	MLENS_HIP_CHECK(hipMemcpy(grads, g_.ptr, nparams_ * sizeof(float), hipMemcpyDeviceToHost));
	return mean_loss(loss.data(), n);
}

void Surrogate::launch_predict(const unsigned short* x, int rows, float* probs)
{
	k_net<false><<<blocks(rows, NET_ROWS), NET_THREADS, 0, stream_>>>(w_.ptr, w16_.ptr, nullptr, x, nullptr, nullptr, rows, probs, nullptr,
		0.0f, NetTrace{});
	MLENS_HIP_CHECK(hipGetLastError());
}

static void pad_inputs(const float* x, int rows, unsigned short* xp)
{
	const size_t padded = size_t(rows + 15) / 16 * 16;
	std::memset(xp, 0, padded * SURR_PIN * sizeof(unsigned short));
	for (int r = 0; r < rows; r++)
		for (int c = 0; c < SURR_NIN; c++) xp[size_t(r) * SURR_PIN + c] = to_bf16(x[size_t(r) * SURR_NIN + c]);
}

/* Requests of up to PREDICT_SMALL rows go through pinned host memory that the kernel reads and writes itself: one
   launch and one wait (a 16-row request spent 30 us in its two copies). Larger ones take PREDICT_ROWS rows at a time
   through device buffers, whose copies are then the smaller cost per byte. */
void Surrogate::predict(const float* x, int n, float* probs)
{
	if (n <= 0) return;
	if (n <= PREDICT_SMALL)
	{
		constexpr size_t in = size_t(PREDICT_SMALL) * SURR_PIN * sizeof(unsigned short);
		if (!small_) MLENS_HIP_CHECK(hipHostMalloc(&small_, in + size_t(PREDICT_SMALL) * SURR_NOUT * sizeof(float), hipHostMallocDefault));
		unsigned short* xp = static_cast<unsigned short*>(small_);
		float* out = reinterpret_cast<float*>(static_cast<char*>(small_) + in);
		pad_inputs(x, n, xp);
		launch_predict(xp, n, out);
		MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
		std::memcpy(probs, out, size_t(n) * SURR_NOUT * sizeof(float));
		return;
	}
	std::vector<unsigned short> xp;
	for (int r0 = 0; r0 < n; r0 += PREDICT_ROWS)
	{
		const int rows = std::min(PREDICT_ROWS, n - r0), M = (rows + 15) / 16 * 16;
		xp.resize(size_t(M) * SURR_PIN);
		pad_inputs(x + size_t(r0) * SURR_NIN, rows, xp.data());
		xb_.alloc(xp.size());
		p_.alloc(size_t(rows) * SURR_NOUT);
		MLENS_HIP_CHECK(hipMemcpyAsync(xb_.ptr, xp.data(), xp.size() * sizeof(unsigned short), hipMemcpyHostToDevice, stream_));
		launch_predict(xb_.ptr, rows, p_.ptr);
		MLENS_HIP_CHECK(hipMemcpyAsync(probs + size_t(r0) * SURR_NOUT, p_.ptr, size_t(rows) * SURR_NOUT * sizeof(float),
			hipMemcpyDeviceToHost, stream_));
		MLENS_HIP_CHECK(hipStreamSynchronize(stream_));
	}
}

double Surrogate::time_predict(const float* x, int n, int reps)
{
	if (n < 1) throw HipError("a timed surrogate request needs at least one row", __FILE__, __LINE__);
	const int rows = std::min(n, max_batch_), M = (rows + 15) / 16 * 16;
	std::vector<unsigned short> xp(size_t(M) * SURR_PIN);
	pad_inputs(x, rows, xp.data());
	xb_.alloc(xp.size());
	p_.alloc(size_t(M) * SURR_NOUT);
	MLENS_HIP_CHECK(hipMemcpyAsync(xb_.ptr, xp.data(), xp.size() * sizeof(unsigned short), hipMemcpyHostToDevice, stream_));
	launch_predict(xb_.ptr, M, p_.ptr);
	hipEvent_t e0, e1;
	MLENS_HIP_CHECK(hipEventCreate(&e0));
	MLENS_HIP_CHECK(hipEventCreate(&e1));
	MLENS_HIP_CHECK(hipEventRecord(e0, stream_));
	for (int r = 0; r < reps; r++) launch_predict(xb_.ptr, M, p_.ptr);
	MLENS_HIP_CHECK(hipEventRecord(e1, stream_));
	MLENS_HIP_CHECK(hipEventSynchronize(e1));
	float ms = 0;
	MLENS_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
	(void)hipEventDestroy(e0);
	(void)hipEventDestroy(e1);
	return ms / 1000.0 / reps / M;   // seconds per predicted histogram
}

}  // namespace mlens
