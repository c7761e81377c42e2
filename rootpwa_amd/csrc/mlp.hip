// mlp.hip -- the learned initializer's network (include/rootpwa_amd_mlp.h).
//
// Products run on FP32 MFMA (v_mfma_f32_16x16x4_f32) with everything that is
// elementwise fused into them: bias, GELU, the loss and its gradient, GELU', the
// bias gradients and Adam.  A training step of L layers is 2 L launches: L
// forward products, L - 1 products dZ W^T, and one launch for the weight
// gradients and the Adam update of all layers.  Every reduction (the K split of
// a product, the sum over a batch's rows, the loss) runs in a fixed order, so
// training is deterministic for a given seed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "internal.h"
#include "rootpwa_amd_mlp.h"

namespace rpwa_amd {
namespace {

constexpr float kInvSqrt2 = 0.70710678118654752440f;
constexpr float kInvSqrt2Pi = 0.39894228040143267794f;

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.f + erff(z * kInvSqrt2)); }

__device__ __forceinline__ float gelu_grad(float z)
{
	return 0.5f * (1.f + erff(z * kInvSqrt2)) + z * kInvSqrt2Pi * expf(-0.5f * z * z);
}

// What bounds a product here: latency.  At the training batch of 64 rows the
// largest one is 64 x 512 x 775 (51 MFLOP, 1.6 MB of weights out of L2): one
// 32 x 32 tile per wave gave 64 waves, each a chain of 388 dependent load /
// MFMA steps (111 us).  So a workgroup owns one 16 x 16 tile (128 workgroups
// there) and its up to kGemmWaves waves split K: wave w takes the 16-deep K groups
// w, w + 8, ..., kGemmDeep of them loaded before the first MFMA, and the waves'
// sums are added in wave order through LDS (5.0 us on average over the hidden
// layers; a training step of the 775 - 3 x 512 - 176 network 730 -> 50 us).
// From kManyTiles tiles on the chip is full and the operands' loads bound a
// product: there a workgroup takes kRowTiles tiles of 16 rows, whose B is loaded
// once (gemm_kernel).
constexpr int kGemmWaves = 8;
constexpr int kGemmThreads = 64 * kGemmWaves;
constexpr int kGemmDeep = 4;  // 16-deep K groups in flight per wave
// Kernels of a forward pass with 1 / kRowTiles tiles per workgroup (with 64 x 64
// tiles of four waves before K was split): 775 - 3 x 512 - 176 at 1024 rows (2048
// tiles in a hidden layer) 70 / 53 us (436), at 256 (512 tiles) 26 / 34 (351), at
// 60000 3.2 / 2.2 ms (4.3); 64 - 2 x 128 - 32 at 4096 rows (2048 tiles) 34 / 18 us
// (51), at 60000 365 / 113 (165); 300 - 1024 - 60 at 256 rows (1024 tiles) 17 / 20 (177).
constexpr int kRowTiles = 4;
constexpr uint32_t kManyTiles = 2048;

typedef float f32x4 __attribute__((ext_vector_type(4)));

enum Epilogue {
	EPI_HIDDEN = 0,  // Z = s + bias, H = GELU(Z)
	EPI_OUT = 1,     // Z = s + bias
	EPI_LOSS = 2,    // dZ = 2 (s + bias - T) / n, the tile's sum of (s + bias - T)^2
	EPI_DZ = 3       // dZ = s GELU'(Z), in the place of Z
};

struct GemmArgs {
	const float* A;         // [M][lda], row r at A + (rowIdx ? rowIdx[r] : r) lda
	const uint32_t* rowIdx;
	const float* B;         // TB ? [N][ldb] : [K][ldb]
	int lda, ldb, M, N, K;
	const float* bias;      // [N]
	float* Z;               // [M][N] pre-activations; dZ with EPI_LOSS and EPI_DZ
	float* H;               // [M][N] activations (EPI_HIDDEN)
	const float* T;         // targets [.][N], row i at T + (tIdx ? tIdx[i] : i) N
	const uint32_t* tIdx;
	float scale;            // 2 / (M N)
	double* tileLoss;       // per workgroup
	uint32_t tile0;         // first workgroup of this launch
};

// workgroups of one launch: a grid has fewer than 2^32 threads
constexpr uint32_t kMaxGrid = 1u << 22;

// 4 consecutive floats at p (aligned to 4 bytes only: rows of any length), zero past `left`
__device__ __forceinline__ f32x4 load4(const float* p, int left)
{
	f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
	if (left >= 4)
		__builtin_memcpy(&v, p, 16);
	else {
		if (left > 0)
			v.x = p[0];
		if (left > 1)
			v.y = p[1];
		if (left > 2)
			v.z = p[2];
	}
	return v;
}

// the first `left` of v's values to p
__device__ __forceinline__ void store4(float* p, const f32x4 v, int left)
{
	if (left >= 4)
		__builtin_memcpy(p, &v, 16);
	else {
		if (left > 0)
			p[0] = v.x;
		if (left > 1)
			p[1] = v.y;
		if (left > 2)
			p[2] = v.z;
	}
}

// C = A op(B) on MT tiles of 16 x 16, one below the other; B's values serve all of
// them, and each tile's sum is the same whatever MT is.  MFMA i of a K group takes
// k = 16 g + 4 q + i in lane quarter q (lane / 16), so a lane's four values are
// consecutive in a row.
template <bool TB, int EPI, int MT>
__global__ __launch_bounds__(kGemmThreads) void gemm_kernel(const GemmArgs a)
{
	__shared__ float red[kGemmWaves][MT * 256];
	// fewer waves where K has fewer groups, but with one tile per workgroup (bound by
	// latency, where the reads of the waves' sums are better known at compile time)
	const int nThreads = MT > 1 ? (int)blockDim.x : kGemmThreads, nWaves = nThreads / 64;
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
	const int r = lane & 15, q = lane >> 4;
	const uint32_t nx = ((uint32_t)a.N + 15) / 16;
	const uint32_t tile = a.tile0 + blockIdx.x;
	const int m0 = (int)(tile / nx) * (16 * MT), n0 = (int)(tile % nx) * 16;
	// rows and columns past the edge repeat the last one; their outputs are not stored
	const int nc = min(n0 + r, a.N - 1);
	const float* pa[MT];
#pragma unroll
	for (int u = 0; u < MT; ++u) {
		const int mc = min(m0 + 16 * u + r, a.M - 1);
		pa[u] = a.A + (size_t)(a.rowIdx ? a.rowIdx[mc] : (uint32_t)mc) * a.lda;
	}
	const float* pb = TB ? a.B + (size_t)nc * a.ldb : a.B + nc;
	const int groups = (a.K + 15) / 16;
	f32x4 acc[MT];
#pragma unroll
	for (int u = 0; u < MT; ++u)
		acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
	constexpr int kDeep = MT > 1 ? 1 : kGemmDeep;
	for (int g0 = wave; g0 < groups; g0 += kGemmWaves * kDeep) {
		f32x4 av[kDeep][MT], bv[kDeep];
#pragma unroll
		for (int d = 0; d < kDeep; ++d) {
			const int g = g0 + d * kGemmWaves, k = 16 * g + 4 * q;
			if (16 * g + 16 <= a.K) {  // the same in every lane
#pragma unroll
				for (int u = 0; u < MT; ++u)
					av[d][u] = load4(pa[u] + k, 4);
				if (TB)
					bv[d] = load4(pb + k, 4);
				else
#pragma unroll
					for (int i = 0; i < 4; ++i)
						bv[d][i] = pb[(size_t)(k + i) * a.ldb];
			} else {  // the last, partial group, and none
				const int left = a.K - k;
#pragma unroll
				for (int u = 0; u < MT; ++u)
					av[d][u] = load4(pa[u] + k, left);
				if (TB)
					bv[d] = load4(pb + k, left);
				else
#pragma unroll
					for (int i = 0; i < 4; ++i)
						bv[d][i] = i < left ? pb[(size_t)(k + i) * a.ldb] : 0.f;
			}
		}
#pragma unroll
		for (int d = 0; d < kDeep; ++d)
#pragma unroll
			for (int i = 0; i < 4; ++i)
#pragma unroll
				for (int u = 0; u < MT; ++u)
					acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[d][u][i], bv[d][i], acc[u], 0, 0, 0);
	}
	// D[i][j]: column j = lane % 16, row i = 4 (lane / 16) + register
#pragma unroll
	for (int u = 0; u < MT; ++u)
#pragma unroll
		for (int v = 0; v < 4; ++v)
			red[wave][256 * u + (4 * q + v) * 16 + r] = acc[u][v];
	__syncthreads();
	double d2 = 0.;
	for (int t = threadIdx.x; t < MT * 256; t += nThreads) {
		float part[kGemmWaves];
#pragma unroll
		for (int w = 0; w < kGemmWaves; ++w)
			part[w] = w < nWaves ? red[w][t] : 0.f;
		float s = part[0];
#pragma unroll
		for (int w = 1; w < kGemmWaves; ++w)
			s += part[w];
		const int i = m0 + t / 16, j = n0 + t % 16;
		if (i < a.M && j < a.N) {
			const size_t o = (size_t)i * a.N + j;
			if (EPI == EPI_DZ) {
				a.Z[o] = s * gelu_grad(a.Z[o]);
			} else {
				const float z = s + a.bias[j];
				if (EPI == EPI_LOSS) {
					const float d = z - a.T[(size_t)(a.tIdx ? a.tIdx[i] : (uint32_t)i) * a.N + j];
					a.Z[o] = a.scale * d;
					d2 += (double)d * (double)d;
				} else {
					a.Z[o] = z;
				}
				if (EPI == EPI_HIDDEN)
					a.H[o] = gelu(z);
			}
		}
	}
	if (EPI == EPI_LOSS) {
		__shared__ double sq[kGemmThreads];
		sq[threadIdx.x] = d2;
		__syncthreads();
		for (int w = min(nThreads, MT * 256) / 2; w > 0; w >>= 1) {
			if ((int)threadIdx.x < w)
				sq[threadIdx.x] += sq[threadIdx.x + w];
			__syncthreads();
		}
		if (threadIdx.x == 0)
			a.tileLoss[tile] = sq[0];
	}
}

// Weight and bias gradients of all layers, and Adam: layer l's parameters are
// the (nIn + 1) x nOut matrix whose last row is the bias, and their gradient is
// [in, 1]^T dZ.  A workgroup owns 16 x 64 parameters: a wave computes 16 x 16
// gradients, and after an exchange through LDS a thread updates four consecutive
// parameters.  Bound by the parameters' and both moments' traffic (24 bytes each,
// read and written: 24 MB at the initializer's size): those loads are in flight
// during the product, and the gradient itself never goes through memory when
// training (10.7 us for the million parameters of the initializer's network; the
// products, column sums and Adam as kernels of their own took 100 us a step).
constexpr int kMaxLayers = 17;
constexpr int kDwDeep = 16;  // rows of the batch per lane quarter in flight

struct DwArgs {
	const float* in[kMaxLayers];   // [rows][nIn] (layer 0: rows through rowIdx)
	const float* dZ[kMaxLayers];   // [rows][nOut]
	int nIn[kMaxLayers], nOut[kMaxLayers];
	uint32_t block0[kMaxLayers + 1];  // first workgroup of each layer
	uint64_t off[kMaxLayers];         // first parameter of each layer
	int nLayers, rows;
	const uint32_t* rowIdx;
	float *p, *m1, *m2;  // Adam; p null: the gradient goes to g
	float* g;
	float lr, c1, c2;
	const double* tileLoss;  // summed in a fixed order by the first wave
	uint32_t nTileLoss;
	double invN;
	float* loss;
	double* epochSum;        // loss added if not null
};

__global__ __launch_bounds__(256) void weight_gradient_kernel(const DwArgs a)
{
	if (blockIdx.x == 0 && threadIdx.x < 64) {
		double s = 0.;
		for (uint32_t k = threadIdx.x; k < a.nTileLoss; k += 64)
			s += a.tileLoss[k];
		for (int d = 32; d >= 1; d >>= 1)
			s += __shfl_xor(s, d);
		if (threadIdx.x == 0) {
			const float l = (float)(s * a.invN);
			*a.loss = l;
			if (a.epochSum)
				*a.epochSum += l;
		}
	}
	int layer = 0;
	while (layer + 1 < a.nLayers && blockIdx.x >= a.block0[layer + 1])
		++layer;
	const int nIn = a.nIn[layer], nOut = a.nOut[layer];
	const uint32_t blk = blockIdx.x - a.block0[layer];
	const uint32_t nx = ((uint32_t)nOut + 63) / 64;
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
	const int r = lane & 15, q = lane >> 4;
	const int m0 = (int)(blk / nx) * 16, n0 = (int)(blk % nx) * 64 + 16 * wave;
	const int m = m0 + r, mc = min(m, nIn - 1), nc = min(n0 + r, nOut - 1);
	const float* in = a.in[layer];
	const float* dZ = a.dZ[layer];
	const uint32_t* rowIdx = layer == 0 ? a.rowIdx : nullptr;
	// this thread's parameters: row i, columns c .. c + 3 (left of them inside the row)
	__shared__ float grad[16][64 + 4];
	const int i = m0 + (int)threadIdx.x / 16, c = (int)(blk % nx) * 64 + 4 * ((int)threadIdx.x % 16);
	const int left = i <= nIn ? nOut - c : 0;
	const size_t o = a.off[layer] + (size_t)i * nOut + c;
	f32x4 p, m1, m2;
	f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
	for (int r0 = 0; r0 < a.rows; r0 += 4 * kDwDeep) {
		// every lane loads (clamped to the edge, so that no branch sits between the
		// loads); rows past the batch are zeroed in both operands, parameter rows and
		// columns past the edge are not stored
		float av[kDwDeep], bv[kDwDeep];
		uint32_t src[kDwDeep];
#pragma unroll
		for (int d = 0; d < kDwDeep; ++d)
			src[d] = (uint32_t)min(r0 + 4 * d + q, a.rows - 1);
#pragma unroll
		for (int d = 0; d < kDwDeep; ++d)
			bv[d] = dZ[(size_t)src[d] * nOut + nc];
		if (rowIdx) {
#pragma unroll
			for (int d = 0; d < kDwDeep; ++d)
				src[d] = rowIdx[src[d]];
		}
#pragma unroll
		for (int d = 0; d < kDwDeep; ++d)
			av[d] = in[(size_t)src[d] * nIn + mc];
		// behind the first operands (loads return in order: in front, the row
		// indices' wait would be theirs too), before the first product
		if (r0 == 0 && a.p) {
			p = load4(a.p + o, left);
			m1 = load4(a.m1 + o, left);
			m2 = load4(a.m2 + o, left);
		}
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int d = 0; d < kDwDeep; ++d) {
			const bool rowOk = r0 + 4 * d + q < a.rows;
			const float x = rowOk ? (m == nIn ? 1.f : av[d]) : 0.f, y = rowOk ? bv[d] : 0.f;
			acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, acc, 0, 0, 0);
		}
	}
#pragma unroll
	for (int v = 0; v < 4; ++v)
		grad[4 * q + v][16 * wave + r] = acc[v];
	__syncthreads();
	f32x4 g;
#pragma unroll
	for (int v = 0; v < 4; ++v)
		g[v] = grad[threadIdx.x / 16][4 * (threadIdx.x % 16) + v];
	if (!a.p) {
		store4(a.g + o, g, left);
		return;
	}
#pragma unroll
	for (int v = 0; v < 4; ++v) {
		m1[v] = 0.9f * m1[v] + 0.1f * g[v];
		m2[v] = 0.999f * m2[v] + 0.001f * g[v] * g[v];
		p[v] -= a.lr * (m1[v] * a.c1) / (sqrtf(m2[v] * a.c2) + 1e-8f);
	}
	store4(a.p + o, p, left);
	store4(a.m1 + o, m1, left);
	store4(a.m2 + o, m2, left);
}

uint64_t mix64(uint64_t x)
{
	x += 0x9E3779B97F4A7C15ull;
	x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
	x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
	return x ^ (x >> 31);
}

}  // namespace
}  // namespace rpwa_amd

using namespace rpwa_amd;

namespace {

// Device copy of a training set.  Up to kKeep bytes stay for the next call (30 us of
// 1500 for an epoch of 1800 x (775 + 176) values, 6.8 MB); a larger one is given back
// at the end of its call.
struct TrainingSet {
	static constexpr size_t kKeep = (size_t)16 << 20;
	float *x = nullptr, *t = nullptr;
	uint32_t* idx = nullptr;
	size_t nX = 0, nT = 0, nIdx = 0;
	~TrainingSet() { release(); }
	bool hold(size_t wantX, size_t wantT, size_t wantIdx)
	{
		if (wantX <= nX && wantT <= nT && wantIdx <= nIdx)
			return true;
		release();
		if (hipMalloc(&x, wantX * sizeof(float)) != hipSuccess || hipMalloc(&t, wantT * sizeof(float)) != hipSuccess ||
		    hipMalloc(&idx, wantIdx * sizeof(uint32_t)) != hipSuccess) {
			release();
			return false;
		}
		nX = wantX, nT = wantT, nIdx = wantIdx;
		return true;
	}
	void release()
	{
		(void)hipFree(x);
		(void)hipFree(t);
		(void)hipFree(idx);
		x = t = nullptr;
		idx = nullptr;
		nX = nT = nIdx = 0;
	}
	// at the end of a call, also a failed one: nothing on the stream uses the set afterwards
	struct Call {
		TrainingSet& set;
		hipStream_t stream;
		~Call()
		{
			(void)hipStreamSynchronize(stream);
			if (sizeof(float) * (set.nX + set.nT + set.nIdx) > kKeep)
				set.release();
		}
	};
};

}  // namespace

struct rpwa_mlp {
	int device = 0;
	std::vector<int> dims;         // nIn, hidden..., nOut
	std::vector<size_t> wOff, bOff;  // parameter offsets
	size_t nParams = 0;
	hipStream_t stream = nullptr;
	float* d_p = nullptr;   // parameters
	float* d_g = nullptr;   // gradient
	float* d_m1 = nullptr;  // Adam moments
	float* d_m2 = nullptr;
	uint64_t adamStep = 0;
	// activations of the current capacity (rows)
	uint32_t capRows = 0;
	std::vector<float*> d_Z, d_H;  // per layer: pre-activation, then its gradient [rows][out]; activation (hidden)
	float* d_x = nullptr;
	float* d_t = nullptr;
	double* d_tileLoss = nullptr;  // per workgroup of the output's product: sum of squared errors
	float* d_loss = nullptr;
	double* d_epoch = nullptr;
	TrainingSet set;

	~rpwa_mlp() { release(); }
	void release_acts()
	{
		for (float* p : d_Z)
			(void)hipFree(p);
		for (float* p : d_H)
			(void)hipFree(p);
		d_Z.clear();
		d_H.clear();
		for (float** p : {&d_x, &d_t})
			if (*p) {
				(void)hipFree(*p);
				*p = nullptr;
			}
		if (d_tileLoss) {
			(void)hipFree(d_tileLoss);
			d_tileLoss = nullptr;
		}
		capRows = 0;
	}
	void release()
	{
		release_acts();
		for (float** p : {&d_p, &d_g, &d_m1, &d_m2, &d_loss})
			if (*p) {
				(void)hipFree(*p);
				*p = nullptr;
			}
		if (d_epoch) {
			(void)hipFree(d_epoch);
			d_epoch = nullptr;
		}
		if (stream) {
			(void)hipStreamDestroy(stream);
			stream = nullptr;
		}
	}
	int nLayers() const { return (int)dims.size() - 1; }
};

namespace {

int check_mlp(const rpwa_mlp* m, const char* fn)
{
	if (!m) {
		set_error(std::string(fn) + ": null network");
		return RPWA_ERR_INVALID;
	}
	return RPWA_OK;
}

// parameters p and zero Adam moments.  On the network's own stream: it does not
// wait for the null stream, so a clear there could run into the next training
int start_state(rpwa_mlp* m, const float* p)
{
	RPWA_HIP_CHECK(hipMemcpyAsync(m->d_p, p, m->nParams * sizeof(float), hipMemcpyHostToDevice, m->stream));
	RPWA_HIP_CHECK(hipMemsetAsync(m->d_m1, 0, m->nParams * sizeof(float), m->stream));
	RPWA_HIP_CHECK(hipMemsetAsync(m->d_m2, 0, m->nParams * sizeof(float), m->stream));
	RPWA_HIP_CHECK(hipStreamSynchronize(m->stream));
	return RPWA_OK;
}

int ensure_rows(rpwa_mlp* m, uint32_t rows)
{
	if (rows <= m->capRows)
		return RPWA_OK;
	m->release_acts();
	const int L = m->nLayers();
	for (int l = 0; l < L; ++l) {
		float *z = nullptr, *h = nullptr;
		RPWA_HIP_CHECK(hipMalloc(&z, (size_t)rows * m->dims[l + 1] * sizeof(float)));
		m->d_Z.push_back(z);
		if (l + 1 < L) {
			RPWA_HIP_CHECK(hipMalloc(&h, (size_t)rows * m->dims[l + 1] * sizeof(float)));
		}
		m->d_H.push_back(h);
	}
	RPWA_HIP_CHECK(hipMalloc(&m->d_x, (size_t)rows * m->dims[0] * sizeof(float)));
	RPWA_HIP_CHECK(hipMalloc(&m->d_t, (size_t)rows * m->dims[L] * sizeof(float)));
	RPWA_HIP_CHECK(hipMalloc(&m->d_tileLoss,
	                         (size_t)((rows + 15) / 16) * ((m->dims[L] + 15) / 16) * sizeof(double)));
	m->capRows = rows;
	return RPWA_OK;
}

// workgroups of an M x N product
struct GemmGrid {
	bool many;
	uint32_t workgroups;
	GemmGrid(int M, int N)
	{
		const uint32_t rowTiles = ((uint32_t)M + 15) / 16, colTiles = ((uint32_t)N + 15) / 16;
		many = (uint64_t)rowTiles * colTiles >= kManyTiles;
		workgroups = (many ? (rowTiles + kRowTiles - 1) / kRowTiles : rowTiles) * colTiles;
	}
};

template <bool TB, int EPI>
int gemm(rpwa_mlp* m, GemmArgs a)
{
	const GemmGrid g(a.M, a.N);
	int waves = g.many ? 1 : kGemmWaves;  // a power of two
	while (waves < kGemmWaves && waves * 16 < a.K)
		waves *= 2;
	for (a.tile0 = 0; a.tile0 < g.workgroups; a.tile0 += std::min(g.workgroups - a.tile0, kMaxGrid)) {
		hipLaunchKernelGGL(g.many ? (gemm_kernel<TB, EPI, kRowTiles>) : (gemm_kernel<TB, EPI, 1>),
		                   dim3(std::min(g.workgroups - a.tile0, kMaxGrid)), dim3(64 * waves), 0, m->stream, a);
		RPWA_HIP_CHECK(hipGetLastError());
	}
	return RPWA_OK;
}

// the rows of a pass: consecutive rows of x (and t), or the rows idx of them
struct Rows {
	const float *x, *t;
	const uint32_t* idx;
	uint32_t n;
};

// forward pass, output in d_Z[L - 1]; withLoss: the loss tiles, and the output's gradient there
int forward(rpwa_mlp* m, const Rows& rows, bool withLoss)
{
	const int L = m->nLayers();
	for (int l = 0; l < L; ++l) {
		GemmArgs a{};
		a.A = l ? m->d_H[l - 1] : rows.x;
		a.rowIdx = l ? nullptr : rows.idx;
		a.B = m->d_p + m->wOff[l];
		a.bias = m->d_p + m->bOff[l];
		a.M = (int)rows.n;
		a.N = a.ldb = m->dims[l + 1];
		a.K = a.lda = m->dims[l];
		a.Z = m->d_Z[l];
		int rc;
		if (l + 1 < L) {
			a.H = m->d_H[l];
			rc = gemm<false, EPI_HIDDEN>(m, a);
		} else if (withLoss) {
			a.T = rows.t;
			a.scale = 2.f / ((float)a.M * (float)a.N);
			a.tileLoss = m->d_tileLoss;
			a.tIdx = rows.idx;
			rc = gemm<false, EPI_LOSS>(m, a);
		} else {
			rc = gemm<false, EPI_OUT>(m, a);
		}
		if (rc != RPWA_OK)
			return rc;
	}
	return RPWA_OK;
}

// Adam of one step
struct AdamStep {
	float lr, c1, c2;
};

// after forward(withLoss): the loss (into d_loss, and added to *epochSum if
// given), and the gradient into d_g or, with adam, straight into the update
int backward(rpwa_mlp* m, const Rows& rows, const AdamStep* adam, double* epochSum)
{
	const int L = m->nLayers();
	for (int l = L - 1; l > 0; --l) {
		// dZ_{l-1} = (dZ_l W_l^T) GELU'(Z_{l-1}), in the place of Z_{l-1}
		GemmArgs a{};
		a.A = m->d_Z[l];
		a.B = m->d_p + m->wOff[l];
		a.M = (int)rows.n;
		a.N = m->dims[l];
		a.K = a.lda = a.ldb = m->dims[l + 1];
		a.Z = m->d_Z[l - 1];
		const int rc = gemm<true, EPI_DZ>(m, a);
		if (rc != RPWA_OK)
			return rc;
	}
	DwArgs d{};
	uint32_t blocks = 0;
	for (int l = 0; l < L; ++l) {
		d.in[l] = l ? m->d_H[l - 1] : rows.x;
		d.dZ[l] = m->d_Z[l];
		d.nIn[l] = m->dims[l];
		d.nOut[l] = m->dims[l + 1];
		d.off[l] = m->wOff[l];
		d.block0[l] = blocks;
		blocks += (uint32_t)((m->dims[l] + 1 + 15) / 16) * (uint32_t)((m->dims[l + 1] + 63) / 64);
	}
	d.block0[L] = blocks;
	d.nLayers = L;
	d.rows = (int)rows.n;
	d.rowIdx = rows.idx;
	if (adam) {
		d.p = m->d_p;
		d.m1 = m->d_m1;
		d.m2 = m->d_m2;
		d.lr = adam->lr;
		d.c1 = adam->c1;
		d.c2 = adam->c2;
	}
	d.g = m->d_g;
	d.tileLoss = m->d_tileLoss;
	d.nTileLoss = GemmGrid((int)rows.n, m->dims[L]).workgroups;
	d.invN = 1. / ((double)rows.n * (double)m->dims[L]);
	d.loss = m->d_loss;
	d.epochSum = epochSum;
	hipLaunchKernelGGL(weight_gradient_kernel, dim3(blocks), dim3(256), 0, m->stream, d);
	RPWA_HIP_CHECK(hipGetLastError());
	return RPWA_OK;
}

}  // namespace

extern "C" int rpwa_mlp_create(rpwa_mlp** out, int device, uint32_t nIn, uint32_t nHidden, uint32_t nHiddenLayers,
                               uint32_t nOut, uint64_t seed)
{
	clear_error();
	if (!out || nIn == 0 || nOut == 0 || (nHiddenLayers > 0 && nHidden == 0) || nHiddenLayers > 16) {
		set_error("rpwa_mlp_create: null pointer or invalid shape");
		return RPWA_ERR_INVALID;
	}
	*out = nullptr;
	int nDev = 0;
	if (hipGetDeviceCount(&nDev) != hipSuccess || device < 0 || device >= nDev) {
		set_error("rpwa_mlp_create: no GPU with index " + std::to_string(device));
		return RPWA_ERR_INVALID;
	}
	std::unique_ptr<rpwa_mlp> m(new rpwa_mlp);
	m->device = device;
	m->dims.push_back((int)nIn);
	for (uint32_t l = 0; l < nHiddenLayers; ++l)
		m->dims.push_back((int)nHidden);
	m->dims.push_back((int)nOut);
	std::vector<float> p;
	for (int l = 0; l < m->nLayers(); ++l) {
		const int nin = m->dims[l], nout = m->dims[l + 1];
		m->wOff.push_back(p.size());
		const double a = std::sqrt(6.0 / (nin + nout));  // Glorot uniform
		for (int k = 0; k < nin * nout; ++k) {
			const uint64_t h = mix64(seed ^ mix64(((uint64_t)l << 40) + (uint64_t)k));
			const double u = ((double)(h >> 11) + 0.5) * (1.0 / 9007199254740992.0);
			p.push_back((float)((2. * u - 1.) * a));
		}
		m->bOff.push_back(p.size());
		p.insert(p.end(), nout, 0.f);
	}
	m->nParams = p.size();
	RPWA_HIP_CHECK(hipSetDevice(device));
	RPWA_HIP_CHECK(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
	RPWA_HIP_CHECK(hipMalloc(&m->d_p, m->nParams * sizeof(float)));
	RPWA_HIP_CHECK(hipMalloc(&m->d_g, m->nParams * sizeof(float)));
	RPWA_HIP_CHECK(hipMalloc(&m->d_m1, m->nParams * sizeof(float)));
	RPWA_HIP_CHECK(hipMalloc(&m->d_m2, m->nParams * sizeof(float)));
	RPWA_HIP_CHECK(hipMalloc(&m->d_loss, sizeof(float)));
	RPWA_HIP_CHECK(hipMalloc(&m->d_epoch, sizeof(double)));
	if (const int rc = start_state(m.get(), p.data()))
		return rc;
	*out = m.release();
	return RPWA_OK;
}

extern "C" int rpwa_mlp_destroy(rpwa_mlp* m)
{
	clear_error();
	if (check_mlp(m, "rpwa_mlp_destroy") != RPWA_OK)
		return RPWA_ERR_INVALID;
	(void)hipSetDevice(m->device);
	if (m->stream)
		(void)hipStreamSynchronize(m->stream);
	delete m;
	return RPWA_OK;
}

extern "C" int rpwa_mlp_nmb_params(const rpwa_mlp* m, uint64_t* n)
{
	clear_error();
	if (check_mlp(m, "rpwa_mlp_nmb_params") != RPWA_OK || !n) {
		set_error("rpwa_mlp_nmb_params: null pointer");
		return RPWA_ERR_INVALID;
	}
	*n = m->nParams;
	return RPWA_OK;
}

extern "C" int rpwa_mlp_get_params(const rpwa_mlp* m, float* params)
{
	clear_error();
	if (check_mlp(m, "rpwa_mlp_get_params") != RPWA_OK || !params) {
		set_error("rpwa_mlp_get_params: null pointer");
		return RPWA_ERR_INVALID;
	}
	RPWA_HIP_CHECK(hipSetDevice(m->device));
	RPWA_HIP_CHECK(hipStreamSynchronize(m->stream));
	RPWA_HIP_CHECK(hipMemcpy(params, m->d_p, m->nParams * sizeof(float), hipMemcpyDeviceToHost));
	return RPWA_OK;
}

extern "C" int rpwa_mlp_set_params(rpwa_mlp* m, const float* params)
{
	clear_error();
	if (check_mlp(m, "rpwa_mlp_set_params") != RPWA_OK || !params) {
		set_error("rpwa_mlp_set_params: null pointer");
		return RPWA_ERR_INVALID;
	}
	RPWA_HIP_CHECK(hipSetDevice(m->device));
	if (const int rc = start_state(m, params))
		return rc;
	m->adamStep = 0;
	return RPWA_OK;
}

extern "C" int rpwa_mlp_forward(rpwa_mlp* m, const float* x, uint32_t nRows, float* y)
{
	clear_error();
	if (check_mlp(m, "rpwa_mlp_forward") != RPWA_OK || !x || !y || nRows == 0) {
		set_error("rpwa_mlp_forward: null pointer or no rows");
		return RPWA_ERR_INVALID;
	}
	RPWA_HIP_CHECK(hipSetDevice(m->device));
	const int rc = ensure_rows(m, nRows);
	if (rc != RPWA_OK)
		return rc;
	RPWA_HIP_CHECK(hipMemcpyAsync(m->d_x, x, (size_t)nRows * m->dims[0] * sizeof(float), hipMemcpyHostToDevice,
	                              m->stream));
	if (forward(m, Rows{m->d_x, nullptr, nullptr, nRows}, false) != RPWA_OK)
		return RPWA_ERR_HIP;
	RPWA_HIP_CHECK(hipMemcpyAsync(y, m->d_Z.back(), (size_t)nRows * m->dims.back() * sizeof(float),
	                              hipMemcpyDeviceToHost, m->stream));
	RPWA_HIP_CHECK(hipStreamSynchronize(m->stream));
	return RPWA_OK;
}

extern "C" int rpwa_mlp_loss_grad(rpwa_mlp* m, const float* x, const float* target, uint32_t nRows, float* loss,
                                  float* grad)
{
	clear_error();
	if (check_mlp(m, "rpwa_mlp_loss_grad") != RPWA_OK || !x || !target || !loss || nRows == 0) {
		set_error("rpwa_mlp_loss_grad: null pointer or no rows");
		return RPWA_ERR_INVALID;
	}
	RPWA_HIP_CHECK(hipSetDevice(m->device));
	int rc = ensure_rows(m, nRows);
	if (rc != RPWA_OK)
		return rc;
	RPWA_HIP_CHECK(hipMemcpyAsync(m->d_x, x, (size_t)nRows * m->dims[0] * sizeof(float), hipMemcpyHostToDevice,
	                              m->stream));
	RPWA_HIP_CHECK(hipMemcpyAsync(m->d_t, target, (size_t)nRows * m->dims.back() * sizeof(float),
	                              hipMemcpyHostToDevice, m->stream));
	const Rows rows{m->d_x, m->d_t, nullptr, nRows};
	if ((rc = forward(m, rows, true)) != RPWA_OK || (rc = backward(m, rows, nullptr, nullptr)) != RPWA_OK)
		return rc;
	RPWA_HIP_CHECK(hipMemcpyAsync(loss, m->d_loss, sizeof(float), hipMemcpyDeviceToHost, m->stream));
	if (grad)
		RPWA_HIP_CHECK(hipMemcpyAsync(grad, m->d_g, m->nParams * sizeof(float), hipMemcpyDeviceToHost, m->stream));
	RPWA_HIP_CHECK(hipStreamSynchronize(m->stream));
	return RPWA_OK;
}

extern "C" int rpwa_mlp_train(rpwa_mlp* m, const float* x, const float* target, uint32_t nRows, uint32_t batchSize,
                              uint32_t nEpochs, float lr, uint64_t seed, float* lossPerEpoch)
{
	clear_error();
	if (check_mlp(m, "rpwa_mlp_train") != RPWA_OK || !x || !target || nRows == 0 || batchSize == 0) {
		set_error("rpwa_mlp_train: null pointer, no rows or zero batch size");
		return RPWA_ERR_INVALID;
	}
	RPWA_HIP_CHECK(hipSetDevice(m->device));
	const uint32_t B = std::min(batchSize, nRows);
	int rc = ensure_rows(m, B);
	if (rc != RPWA_OK)
		return rc;
	const int nIn = m->dims[0], nOut = m->dims.back();
	TrainingSet& set = m->set;
	const TrainingSet::Call call{set, m->stream};
	if (!set.hold((size_t)nRows * nIn, (size_t)nRows * nOut, nRows)) {
		set_error("rpwa_mlp_train: device allocation failed");
		return RPWA_ERR_NOMEM;
	}
	if (hipMemcpyAsync(set.x, x, (size_t)nRows * nIn * sizeof(float), hipMemcpyHostToDevice, m->stream) != hipSuccess ||
	    hipMemcpyAsync(set.t, target, (size_t)nRows * nOut * sizeof(float), hipMemcpyHostToDevice, m->stream) !=
	        hipSuccess ||
	    hipStreamSynchronize(m->stream) != hipSuccess) {
		set_error("rpwa_mlp_train: copy failed");
		return RPWA_ERR_HIP;
	}
	std::vector<uint32_t> perm(nRows);
	for (uint32_t epoch = 0; epoch < nEpochs && rc == RPWA_OK; ++epoch) {
		// Fisher-Yates shuffle from counter-based draws
		for (uint32_t i = 0; i < nRows; ++i)
			perm[i] = i;
		for (uint32_t i = nRows - 1; i > 0; --i) {
			const uint64_t h = mix64(seed ^ mix64(((uint64_t)epoch << 32) + i));
			std::swap(perm[i], perm[(uint32_t)(h % (i + 1))]);
		}
		if (hipMemcpyAsync(set.idx, perm.data(), nRows * sizeof(uint32_t), hipMemcpyHostToDevice, m->stream) !=
		        hipSuccess ||
		    hipMemsetAsync(m->d_epoch, 0, sizeof(double), m->stream) != hipSuccess) {
			rc = RPWA_ERR_HIP;
			break;
		}
		const uint32_t nBatches = nRows / B;  // full batches only
		for (uint32_t bi = 0; bi < nBatches && rc == RPWA_OK; ++bi) {
			++m->adamStep;
			const AdamStep adam{lr, (float)(1. / (1. - std::pow(0.9, (double)m->adamStep))),
			                    (float)(1. / (1. - std::pow(0.999, (double)m->adamStep)))};
			const Rows rows{set.x, set.t, set.idx + (size_t)bi * B, B};
			if ((rc = forward(m, rows, true)) == RPWA_OK)
				rc = backward(m, rows, &adam, m->d_epoch);
		}
		if (rc == RPWA_OK && lossPerEpoch) {
			double s = 0.;
			if (hipMemcpyAsync(&s, m->d_epoch, sizeof(double), hipMemcpyDeviceToHost, m->stream) != hipSuccess ||
			    hipStreamSynchronize(m->stream) != hipSuccess)
				rc = RPWA_ERR_HIP;
			lossPerEpoch[epoch] = (float)(s / std::max(nBatches, 1u));
		}
	}
	if (hipStreamSynchronize(m->stream) != hipSuccess && rc == RPWA_OK)
		rc = RPWA_ERR_HIP;
	if (rc != RPWA_OK && rpwa_last_error()[0] == 0)
		set_error("rpwa_mlp_train: a kernel launch or copy failed");
	return rc;
}
