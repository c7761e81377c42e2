// integral.hip -- A.A^dagger normalisation integrals on FP64 MFMA (gfx950).
//
// ampIntegralMatrix::integrate (decayAmplitude/ampIntegralMatrix.cc:408-483)
// accumulates I_ij = sum_e wt_e A_i(e) conj(A_j(e)).  With the amplitude row of
// an event read as the real vector x_e = (Re A_0, Im A_0, Re A_1, ...) of length
// D = 2W (the interleaved complex128 row, no copy), the real symmetric matrix
//   C = sum_e wt_e x_e x_e^T                      (D x D)
// holds every product:
//   Re I_ij = C[2i][2j] + C[2i+1][2j+1],   Im I_ij = C[2i+1][2j] - C[2i][2j+1].
// C is computed as a rank-k update on v_mfma_f64_16x16x4_f64 (rank_update.h): 16x16
// output tiles of the upper triangle (tile row <= tile column), k = events.  Each
// workgroup writes its tile sums to a partial row; partial rows are summed in
// fixed order (column_sum_kernel), and the host assembles the complex matrix.
#include "internal.h"
#include "rank_update.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

namespace rpwa_amd {
namespace {

// fixed-order column sums of a [nRows][nCols] array
constexpr int kColElems = 64;
constexpr int kColChunks = 16;
__global__ __launch_bounds__(kColElems* kColChunks) void column_sum_kernel(
    const double* __restrict__ in, int nRows, uint32_t nCols, double* __restrict__ out)
{
	__shared__ double sh[kColChunks][kColElems];
	const int el = threadIdx.x % kColElems;
	const int ch = threadIdx.x / kColElems;
	const uint32_t col = blockIdx.x * kColElems + el;
	const int r0 = (int)((int64_t)nRows * ch / kColChunks);
	const int r1 = (int)((int64_t)nRows * (ch + 1) / kColChunks);
	double s = 0.;
	if (col < nCols)
		for (int r = r0; r < r1; ++r)
			s += in[(size_t)r * nCols + col];
	sh[ch][el] = s;
	__syncthreads();
	if (ch == 0 && col < nCols) {
		double t = 0.;
		for (int k = 0; k < kColChunks; ++k)
			t += sh[k][el];
		out[col] = t;
	}
}

}  // namespace

hipError_t launch_column_sum(const double* in, int nRows, uint32_t nCols, double* out, hipStream_t s)
{
	hipLaunchKernelGGL(column_sum_kernel, dim3((nCols + kColElems - 1) / kColElems), dim3(kColElems * kColChunks), 0, s,
	                   in, nRows, nCols, out);
	return hipGetLastError();
}

// partial tiles of n rows of D doubles (D even)
static hipError_t launch_rows(const double* x, const double* w, bool direct, uint64_t n, uint32_t D, double* partials,
                              double* wsum, bool accumulate, int nWg, hipStream_t s)
{
	ru::Args a{};
	a.x = x;
	a.w = w;
	a.n = n;
	a.D = D;
	a.partials = partials;
	a.wsum = wsum;
	a.accumulate = accumulate ? 1 : 0;
	a.direct = direct ? 1 : 0;
	return w ? ru::launch<true>(a, nWg, s) : ru::launch<false>(a, nWg, s);
}

struct IntegralPlan {
	uint32_t nT, nTiles;
	int nWg;
};

// D = real row length (2 x complex values per row); one workgroup per CU
static int integral_plan(int device, uint32_t D, IntegralPlan& p)
{
	p.nT = (D + 15) / 16;
	p.nTiles = p.nT * (p.nT + 1) / 2;
	int nCu = 0;
	RPWA_HIP_CHECK(hipDeviceGetAttribute(&nCu, hipDeviceAttributeMultiprocessorCount, device));
	p.nWg = nCu > 0 ? nCu : 1;
	return RPWA_OK;
}

// Per-device work area of the rank-k update (workgroup partial tiles, weight
// sums, reduced tiles) and its stream, kept between calls and grown on demand:
// a call then allocates nothing of its own on the device (an allocation and a
// free of the ~35 MB partials, with the free's device synchronisation, cost
// about as much as a tenth of the update at 5M x 88).  Calls on one device are
// serialised by the mutex; the area lives until the process ends.
struct SyrkWork {
	std::mutex m;
	hipStream_t s = nullptr;
	double* part = nullptr;
	double* wsum = nullptr;
	double* red = nullptr;
	size_t partCap = 0, wsumCap = 0, redCap = 0;
};
constexpr int kSyrkDevices = 64;

static SyrkWork& syrk_work(int device)
{
	static SyrkWork work[kSyrkDevices];
	return work[device];
}

static hipError_t syrk_grow(double*& buf, size_t& cap, size_t need)
{
	if (need <= cap)
		return hipSuccess;
	if (buf)
		(void)hipFree(buf);
	buf = nullptr;
	cap = 0;
	hipError_t e = hipMalloc(&buf, need * sizeof(double));
	if (e == hipSuccess)
		cap = need;
	return e;
}

// Weighted real rank-k update C = sum_e wt_e x_e x_e^T of M rows of D doubles
// (device or host memory); wt_e = w[e] (directWeights) or 1/w[e] or 1.
// Returns the full symmetric D x D matrix and the sum of the weights.
static int syrk_run(int device, const double* d_x, uint64_t M, uint32_t D, const double* d_w, bool directWeights,
             const double* h_x, const double* h_w, std::vector<double>& full, double* wtot)
{
	if (device < 0 || device >= kSyrkDevices) {
		set_error("rank-k update: device index out of range");
		return RPWA_ERR_INVALID;
	}
	RPWA_HIP_CHECK(hipSetDevice(device));
	const bool weighted = (d_w != nullptr) || (h_w != nullptr);
	IntegralPlan p;
	int st = integral_plan(device, D, p);
	if (st != RPWA_OK)
		return st;
	SyrkWork& work = syrk_work(device);
	std::lock_guard<std::mutex> lock(work.m);
	if (!work.s)
		RPWA_HIP_CHECK(hipStreamCreateWithFlags(&work.s, hipStreamNonBlocking));
	hipStream_t s = work.s;
	double* d_stage[2] = {nullptr, nullptr};
	double* d_wstage[2] = {nullptr, nullptr};
	const size_t partN = (size_t)p.nWg * p.nTiles * 256;
	std::vector<double> C((size_t)p.nTiles * 256);
	std::vector<double> wsums(p.nWg);
	auto fail = [&](int code) {
		if (code != RPWA_OK)
			(void)hipStreamSynchronize(s);  // nothing of this call may still run on the work area
		(void)hipFree(d_stage[0]); (void)hipFree(d_stage[1]); (void)hipFree(d_wstage[0]); (void)hipFree(d_wstage[1]);
		return code;
	};
#define INT_CHECK(expr)                                                               \
	do {                                                                              \
		hipError_t e_ = (expr);                                                       \
		if (e_ != hipSuccess) {                                                       \
			set_error(std::string(#expr) + ": " + hipGetErrorString(e_));             \
			return fail(RPWA_ERR_HIP);                                                \
		}                                                                             \
	} while (0)
	INT_CHECK(syrk_grow(work.part, work.partCap, partN));
	INT_CHECK(syrk_grow(work.wsum, work.wsumCap, p.nWg));
	INT_CHECK(syrk_grow(work.red, work.redCap, (size_t)p.nTiles * 256));
	double* d_part = work.part;
	double* d_wsum = work.wsum;
	double* d_red = work.red;
	if (d_x) {
		INT_CHECK(launch_rows(d_x, d_w, directWeights, M, D, d_part, d_wsum, false, p.nWg, s));
	} else {
		// stream the host array through two device buffers
		const uint64_t chunkEv = std::max<uint64_t>(1, (256ull << 20) / (8ull * D));
		for (int b = 0; b < 2; ++b) {
			INT_CHECK(hipMalloc(&d_stage[b], chunkEv * 8ull * D));
			if (weighted)
				INT_CHECK(hipMalloc(&d_wstage[b], chunkEv * sizeof(double)));
		}
		hipEvent_t done[2];
		INT_CHECK(hipEventCreate(&done[0]));
		INT_CHECK(hipEventCreate(&done[1]));
		bool first = true;
		int b = 0;
		for (uint64_t off = 0; off < M; off += chunkEv, b ^= 1) {
			const uint64_t n = std::min<uint64_t>(chunkEv, M - off);
			if (!first)
				INT_CHECK(hipEventSynchronize(done[b]));
			INT_CHECK(hipMemcpyAsync(d_stage[b], h_x + off * D, n * 8ull * D, hipMemcpyHostToDevice, s));
			if (weighted)
				INT_CHECK(hipMemcpyAsync(d_wstage[b], h_w + off, n * sizeof(double), hipMemcpyHostToDevice, s));
			INT_CHECK(launch_rows(d_stage[b], weighted ? d_wstage[b] : nullptr, directWeights, n, D, d_part, d_wsum, !first,
			                      p.nWg, s));
			INT_CHECK(hipEventRecord(done[b], s));
			first = false;
		}
		INT_CHECK(hipStreamSynchronize(s));
		(void)hipEventDestroy(done[0]);
		(void)hipEventDestroy(done[1]);
	}
	INT_CHECK(launch_column_sum(d_part, p.nWg, p.nTiles * 256, d_red, s));
	INT_CHECK(hipMemcpyAsync(C.data(), d_red, C.size() * sizeof(double), hipMemcpyDeviceToHost, s));
	if (weighted)
		INT_CHECK(hipMemcpyAsync(wsums.data(), d_wsum, wsums.size() * sizeof(double), hipMemcpyDeviceToHost, s));
	INT_CHECK(hipStreamSynchronize(s));
#undef INT_CHECK
	// the symmetric matrix from the upper-triangle tiles, tile by tile: a
	// diagonal tile as computed (with weights its two halves can differ in the
	// last bit), an off-diagonal tile at (I, J) and transposed at (J, I)
	full.assign((size_t)D * D, 0.);
	for (uint32_t I = 0, t = 0; I < p.nT; ++I)
		for (uint32_t J = I; J < p.nT; ++J, ++t) {
			const double* tile = C.data() + (size_t)t * 256;
			const uint32_t r1 = std::min<uint32_t>(16, D - 16 * I), c1 = std::min<uint32_t>(16, D - 16 * J);
			for (uint32_t r = 0; r < r1; ++r)
				for (uint32_t c = 0; c < c1; ++c) {
					const uint32_t row = 16 * I + r, col = 16 * J + c;
					full[(size_t)row * D + col] = tile[r * 16 + c];
					if (I != J)
						full[(size_t)col * D + row] = tile[r * 16 + c];
				}
		}
	if (wtot) {
		double t = weighted ? 0. : (double)M;
		for (double v : wsums)
			t += v;
		*wtot = t;
	}
	fail(RPWA_OK);
	return RPWA_OK;
}

static int integral_run(int device, const double* d_amps, uint64_t M, uint32_t W, const double* d_w,
                        double* outSums, const double* h_amps, const double* h_w)
{
	std::vector<double> C;
	double wtot = 0.;
	const uint32_t D = 2 * W;
	int st = syrk_run(device, d_amps, M, D, d_w, false, h_amps, h_w, C, &wtot);
	if (st != RPWA_OK)
		return st;
	for (uint32_t i = 0; i < W; ++i)
		for (uint32_t j = 0; j < W; ++j) {
			const double re = C[(size_t)(2 * i) * D + 2 * j] + C[(size_t)(2 * i + 1) * D + 2 * j + 1];
			const double im = C[(size_t)(2 * i + 1) * D + 2 * j] - C[(size_t)(2 * i) * D + 2 * j + 1];
			outSums[2 * ((size_t)i * W + j)] = re;
			outSums[2 * ((size_t)i * W + j) + 1] = im;
		}
	if (d_w || h_w) {
		// renormalise to the weight integral (ampIntegralMatrix.cc:477-483)
		const double weightNorm = wtot / (double)M;
		const double inv = 1 / weightNorm;
		for (size_t i = 0; i < (size_t)2 * W * W; ++i)
			outSums[i] *= inv;
	}
	return RPWA_OK;
}

// per event w_e = 1 / sum_i |A_i(e)|^2 / I_ii (0 for an all-zero event)
__global__ void inverse_norm_kernel(const double2* __restrict__ amps, uint64_t M, uint32_t W,
                                    const double* __restrict__ invDiag, double* __restrict__ w)
{
	const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (e >= M)
		return;
	double s = 0.;
	for (uint32_t i = 0; i < W; ++i) {
		const double2 a = amps[e * W + i];
		s += (a.x * a.x + a.y * a.y) * invDiag[i];
	}
	w[e] = s > 0. ? 1. / s : 0.;
}

static int moments_run(int device, const double* d_amps, uint64_t M, uint32_t W, const double* normDiag,
                       int perEventNorm, double* out)
{
	std::vector<double> C;
	double wtot = 0.;
	const uint32_t D = 2 * W;
	double* d_w = nullptr;
	double* d_inv = nullptr;
	std::vector<double> inv(W);
	for (uint32_t i = 0; i < W; ++i)
		inv[i] = normDiag[i] > 0. ? 1. / normDiag[i] : 0.;
	if (perEventNorm) {
		RPWA_HIP_CHECK(hipSetDevice(device));
		RPWA_HIP_CHECK(hipMalloc(&d_w, M * sizeof(double)));
		if (hipMalloc(&d_inv, W * sizeof(double)) != hipSuccess ||
		    hipMemcpy(d_inv, inv.data(), W * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
			(void)hipFree(d_w);
			if (d_inv)
				(void)hipFree(d_inv);
			set_error("rpwa_data_moments_device: allocation or copy failed");
			return RPWA_ERR_HIP;
		}
		hipLaunchKernelGGL(inverse_norm_kernel, dim3((uint32_t)((M + 255) / 256)), dim3(256), 0, 0,
		                   reinterpret_cast<const double2*>(d_amps), M, W, d_inv, d_w);
		const hipError_t e = hipDeviceSynchronize();
		(void)hipFree(d_inv);
		if (e != hipSuccess) {
			(void)hipFree(d_w);
			set_error(std::string("rpwa_data_moments_device: ") + hipGetErrorString(e));
			return RPWA_ERR_HIP;
		}
	}
	const int st = syrk_run(device, d_amps, M, D, d_w, true, nullptr, nullptr, C, &wtot);
	if (d_w)
		(void)hipFree(d_w);
	if (st != RPWA_OK)
		return st;
	for (uint32_t i = 0; i < W; ++i)
		for (uint32_t j = 0; j < W; ++j) {
			const double re = C[(size_t)(2 * i) * D + 2 * j] + C[(size_t)(2 * i + 1) * D + 2 * j + 1];
			const double im = C[(size_t)(2 * i + 1) * D + 2 * j] - C[(size_t)(2 * i) * D + 2 * j + 1];
			const double sc = std::sqrt(inv[i] * inv[j]) / (double)M;
			out[2 * ((size_t)i * W + j)] = re * sc;
			out[2 * ((size_t)i * W + j) + 1] = im * sc;
		}
	return RPWA_OK;
}

// ---------------------------------------------------------------------------
// The integral without allocations (rpwa_integral_device_noalloc): the same
// kernels and reduction order as integral_run on device input, with every
// intermediate in one static device array instead of hipMalloc'd buffers.
// Layout of the array (doubles): workgroup partial tiles
// [kNaWg][kNaTiles][256], workgroup weight sums [kNaWg], reduced tiles
// [kNaTiles][256], the complex result [W][W].  Every element a call reads is
// written earlier in the same call, so nothing needs clearing between calls.
constexpr uint32_t kNaMaxWaves = 128;                       // D = 256: 16 x 16 tiles of 16 x 16
constexpr uint32_t kNaTiles = (2 * kNaMaxWaves / 16) * (2 * kNaMaxWaves / 16 + 1) / 2;  // 136
constexpr int kNaWg = 256;                                  // one workgroup per CU of an MI355X
constexpr size_t kNaPartial = (size_t)kNaWg * kNaTiles * 256;
constexpr size_t kNaWsum = kNaPartial;
constexpr size_t kNaRed = kNaWsum + kNaWg;
constexpr size_t kNaOut = kNaRed + (size_t)kNaTiles * 256;
constexpr size_t kNaDoubles = kNaOut + 2ull * kNaMaxWaves * kNaMaxWaves;  // 8,980,736 doubles = 68.5 MiB
constexpr int kNaMaxDevices = 64;

static __device__ __align__(256) double scratch[kNaDoubles];

namespace {

// per-device address of `scratch`, looked up once per device with that device current
std::once_flag g_naOnce[kNaMaxDevices];
double* g_naPtr[kNaMaxDevices];
hipError_t g_naErr[kNaMaxDevices];

// the complex sums [W][W] from the reduced tiles (the host assembly of integral_run),
// renormalised by the mean weight when weights are given (ampIntegralMatrix.cc:477-483)
__global__ __launch_bounds__(256) void assemble_kernel(const double* __restrict__ red, uint32_t nT, uint32_t W,
                                                       const double* __restrict__ wsum, int nWg, uint64_t M,
                                                       int weighted, double* __restrict__ out)
{
	const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
	if (idx >= W * W)
		return;
	const uint32_t i = idx / W, j = idx % W;
	auto c = [&](uint32_t r, uint32_t col) {
		uint32_t I = r / 16, J = col / 16;
		if (I > J) {
			const uint32_t t = r;
			r = col;
			col = t;
			const uint32_t u = I;
			I = J;
			J = u;
		}
		const uint32_t t = I * nT - I * (I - 1) / 2 + (J - I);
		return red[(size_t)t * 256 + (r % 16) * 16 + (col % 16)];
	};
	double re = c(2 * i, 2 * j) + c(2 * i + 1, 2 * j + 1);
	double im = c(2 * i + 1, 2 * j) - c(2 * i, 2 * j + 1);
	if (weighted) {
		double t = 0.;
		for (int r = 0; r < nWg; ++r)
			t += wsum[r];
		const double weightNorm = t / (double)M;
		const double inv = 1 / weightNorm;
		re *= inv;
		im *= inv;
	}
	out[2 * (size_t)idx] = re;
	out[2 * (size_t)idx + 1] = im;
}

}  // namespace

static int integral_noalloc(int device, const double* d_amps, uint64_t M, uint32_t W, const double* d_w,
                            double* outSums)
{
	if (W > kNaMaxWaves) {
		set_error("rpwa_integral_device_noalloc: " + std::to_string(W) + " waves exceed the static work area (at "
		          "most " + std::to_string(kNaMaxWaves) + "); use rpwa_integral_device");
		return RPWA_ERR_UNSUPPORTED;
	}
	int nDev = 0;
	RPWA_HIP_CHECK(hipGetDeviceCount(&nDev));
	if (device < 0 || device >= nDev || device >= kNaMaxDevices) {
		set_error("rpwa_integral_device_noalloc: no GPU with index " + std::to_string(device));
		return RPWA_ERR_INVALID;
	}
	RPWA_HIP_CHECK(hipSetDevice(device));
	std::call_once(g_naOnce[device], [device]() {
		g_naErr[device] = hipGetSymbolAddress(reinterpret_cast<void**>(&g_naPtr[device]), HIP_SYMBOL(scratch));
	});
	if (g_naErr[device] != hipSuccess || !g_naPtr[device]) {
		set_error(std::string("rpwa_integral_device_noalloc: hipGetSymbolAddress(scratch): ") +
		          hipGetErrorString(g_naErr[device]));
		return RPWA_ERR_HIP;
	}
	double* const base = g_naPtr[device];
	const bool weighted = d_w != nullptr;
	IntegralPlan p;
	if (int st = integral_plan(device, 2 * W, p))
		return st;
	p.nWg = std::min(p.nWg, kNaWg);
	RPWA_HIP_CHECK(launch_rows(d_amps, d_w, false, M, 2 * W, base, base + kNaWsum, false, p.nWg, 0));
	RPWA_HIP_CHECK(launch_column_sum(base, p.nWg, p.nTiles * 256, base + kNaRed, 0));
	hipLaunchKernelGGL(assemble_kernel, dim3((W * W + 255) / 256), dim3(256), 0, 0, base + kNaRed, p.nT, W,
	                   base + kNaWsum, p.nWg, M, weighted ? 1 : 0, base + kNaOut);
	RPWA_HIP_CHECK(hipGetLastError());
	RPWA_HIP_CHECK(hipMemcpy(outSums, base + kNaOut, (size_t)W * W * 2 * sizeof(double), hipMemcpyDeviceToHost));
	return RPWA_OK;
}

}  // namespace rpwa_amd

extern "C" int rpwa_integral_device_noalloc(int device, const double* d_amps, uint64_t nmbEvents,
                                            uint32_t nmbWaves, const double* d_weights, double* outSums)
{
	rpwa_amd::clear_error();
	if (!d_amps || !outSums || nmbEvents == 0 || nmbWaves == 0) {
		rpwa_amd::set_error("rpwa_integral_device_noalloc: null pointer or empty input");
		return RPWA_ERR_INVALID;
	}
	try {
		return rpwa_amd::integral_noalloc(device, d_amps, nmbEvents, nmbWaves, d_weights, outSums);
	} catch (const std::exception& ex) {
		rpwa_amd::set_error(ex.what());
		return RPWA_ERR_INVALID;
	}
}

extern "C" int rpwa_data_moments_device(int device, const double* d_amps, uint64_t nmbEvents, uint32_t nmbWaves,
                                        const double* normDiag, int perEventNorm, double* outMoments)
{
	rpwa_amd::clear_error();
	if (!d_amps || !normDiag || !outMoments || nmbEvents == 0 || nmbWaves == 0) {
		rpwa_amd::set_error("rpwa_data_moments_device: null pointer or empty input");
		return RPWA_ERR_INVALID;
	}
	try {
		return rpwa_amd::moments_run(device, d_amps, nmbEvents, nmbWaves, normDiag, perEventNorm, outMoments);
	} catch (const std::exception& ex) {
		rpwa_amd::set_error(ex.what());
		return RPWA_ERR_NOMEM;
	}
}

extern "C" int rpwa_integral(int device, const double* amps, uint64_t nmbEvents, uint32_t nmbWaves,
                             const double* weights, double* outSums)
{
	rpwa_amd::clear_error();
	if (!amps || !outSums || nmbEvents == 0 || nmbWaves == 0) {
		rpwa_amd::set_error("rpwa_integral: null pointer or empty input");
		return RPWA_ERR_INVALID;
	}
	try {
		return rpwa_amd::integral_run(device, nullptr, nmbEvents, nmbWaves, nullptr, outSums, amps,
		                              weights);
	} catch (const std::exception& ex) {
		rpwa_amd::set_error(ex.what());
		return RPWA_ERR_NOMEM;
	}
}

extern "C" int rpwa_integral_device(int device, const double* d_amps, uint64_t nmbEvents,
                                    uint32_t nmbWaves, const double* d_weights, double* outSums)
{
	rpwa_amd::clear_error();
	if (!d_amps || !outSums || nmbEvents == 0 || nmbWaves == 0) {
		rpwa_amd::set_error("rpwa_integral_device: null pointer or empty input");
		return RPWA_ERR_INVALID;
	}
	try {
		return rpwa_amd::integral_run(device, d_amps, nmbEvents, nmbWaves, d_weights, outSums,
		                              nullptr, nullptr);
	} catch (const std::exception& ex) {
		rpwa_amd::set_error(ex.what());
		return RPWA_ERR_NOMEM;
	}
}
