// hessian.hip -- event part of the analytic Hessian on the GPU.
//
// pwaLikelihood::Hessian (partialWaveFit/pwaLikelihood.cc:697-753) sums per event
//   factor2 * Re/Im(d_b) * Re/Im(d_a)            with d_a = S_{r_a s_a}(e) conj(A_a(e)),
//   - factor * Re/Im(A_a conj(A_b))               for a, b of the same (rank, sector),
//   factor2 * flat * d_a  and  factor2 * flat^2 - factor,
// factor = 2 / sigma_e, factor2 = factor^2.  The first two are rank-k updates over
// events, sum_e x x^T of the real rows x = factor d (2 R rowLen doubles) and x =
// sqrt(factor) A (2 rowLen), on v_mfma_f64_16x16x4_f64.  A first kernel computes S and
// the weights of every event; the rank-k passes then form the rows from S and
// the stored amplitudes while they copy a chunk of events into LDS, so that no
// row array goes through memory.  The flat wave's terms are column sums of factor2
// d, taken by the threads that form d, and sums of the factors.
// 2M events x 88 waves x rank 2, complex64 amplitudes: 9.98 -> 7.16 ms; before, a
// kernel wrote the rows (8.5 GB, 2.3 ms) and weighted passes read them (7.1 ms).
#include "event_kernel.h"
#include "hessian_pass.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

namespace rpwa_amd {
namespace {

template <bool MIXED>
__device__ __forceinline__ double2 amp_at(const void* amps, uint64_t i)
{
	if (MIXED) {
		const float2 v = reinterpret_cast<const float2*>(amps)[i];
		return make_double2((double)v.x, (double)v.y);
	}
	return reinterpret_cast<const double2*>(amps)[i];
}

// factor S of every (rank, sector), factor and sqrt(factor) of every event: with
// the rows scaled on both sides the products need no weights (FP64 vector
// multiplies take the matrix core's turns).  L lanes per event, T [rank][rowLen]
// (zero on padding) from the caches.  Bound by one read of the amplitudes
// (2M x 88 complex64: 0.38 ms, 3.8 TB/s), and in narrow rows by the sums over an
// event's lanes, which are the same for any row length: 4 lanes there.
template <bool MIXED, uint32_t L>
__global__ __launch_bounds__(256) void hessian_s_kernel(const void* amps, uint64_t e0, uint64_t n, uint32_t rowLen,
                                                        uint32_t secOff1, uint32_t rank,
                                                        const double2* __restrict__ T, double flat2,
                                                        double2* __restrict__ S, double* __restrict__ wD,
                                                        double* __restrict__ wA)
{
	// per group of L lanes kE events at a time: their loads are in flight together
	// and share the loads of T
	constexpr uint32_t kR = 2, kE = L / 4;
	const uint32_t lig = threadIdx.x % L, grp = (threadIdx.x % 64) / L;
	const uint64_t stride = (uint64_t)gridDim.x * (256 / L * kE);
	// the loop's bound is the same in a wave's groups (16 events): the sums below take all lanes
	for (uint64_t first = ((uint64_t)blockIdx.x * 4 + threadIdx.x / 64) * 16; first < n; first += stride) {
		uint64_t row[kE];
		double sigma[kE];
#pragma unroll
		for (uint32_t i = 0; i < kE; ++i) {
			row[i] = (e0 + min(first + kE * grp + i, n - 1)) * rowLen;
			sigma[i] = 0.;
		}
		// lane lig of a group writes S of event lig / 4, rank r0 + (lig / 2) % 2, sector lig % 2
		const uint64_t mineEv = first + kE * grp + lig / 4;
		double2 mine;
		for (uint32_t r0 = 0;; r0 += kR) {
			const bool two = r0 + 1 < rank;
#pragma unroll
			for (uint32_t s = 0; s < 2; ++s) {
				const uint32_t c0 = s ? secOff1 : 0, c1 = s ? rowLen : secOff1;
				double2 acc[kE][kR];
#pragma unroll
				for (uint32_t i = 0; i < kE; ++i)
#pragma unroll
					for (uint32_t r = 0; r < kR; ++r)
						acc[i][r] = make_double2(0., 0.);
#pragma unroll 2
				for (uint32_t c = c0 + lig; c < c1; c += L) {
					const double2 t0 = T[(size_t)r0 * rowLen + c], t1 = T[(size_t)(two ? r0 + 1 : r0) * rowLen + c];
#pragma unroll
					for (uint32_t i = 0; i < kE; ++i) {
						const double2 x = amp_at<MIXED>(amps, row[i] + c);
						ek::cmac(acc[i][0], t0, x);
						ek::cmac(acc[i][1], t1, x);
					}
				}
#pragma unroll
				for (uint32_t i = 0; i < kE; ++i)
#pragma unroll
					for (uint32_t r = 0; r < kR; ++r) {
						const double2 v = make_double2(ek::group_sum<(int)L>(acc[i][r].x), ek::group_sum<(int)L>(acc[i][r].y));
						if (r == 0 || two)
							sigma[i] += v.x * v.x + v.y * v.y;
						if (lig == 4 * i + 2 * r + s)
							mine = v;
					}
			}
			if (r0 + kR >= rank) {
				// sigma is complete: this block's S and, for ranks above 2, the earlier ones
				double f = 0.;
#pragma unroll
				for (uint32_t i = 0; i < kE; ++i) {
					const double factor = 2. / (sigma[i] + flat2);
					if (lig / 4 == i)
						f = factor;
				}
				if (mineEv < n) {
					double2* o = S + mineEv * 2 * rank + lig % 4;
					for (uint32_t q = 0; q < r0; q += kR)
						o[2 * q] = make_double2(o[2 * q].x * f, o[2 * q].y * f);
					if (lig % 4 < 2 || two)
						o[2 * r0] = make_double2(mine.x * f, mine.y * f);
					if (lig % 4 == 0) {
						wD[mineEv] = f;
						wA[mineEv] = sqrt(f);
					}
				}
				break;
			}
			if (mineEv < n)
				S[mineEv * 2 * rank + 2 * r0 + lig % 4] = mine;
		}
	}
}

// Longest row that takes 4 lanes per event.  A call with 4 / 16 lanes, us: 1M events x
// 4 columns x rank 1 211 / 290, x 24 x rank 2 591 / 646, 300k x 40 x rank 1 281 / 286,
// x 54 x rank 3 1252 / 1212.
constexpr uint32_t kNarrow = 40;

// Per-device work area of the Hessian (S and the weights of the events, T, the
// workgroups' sums), kept between calls and grown on demand: a call then
// allocates nothing on the device.  Calls on one device are serialised by the
// mutex; the area lives until the process ends.
struct HessWork {
	std::mutex m;
	char* buf = nullptr;
	size_t cap = 0;
};
constexpr int kHessDevices = 64;

HessWork& hess_work(int device)
{
	static HessWork work[kHessDevices];
	return work[device];
}

constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace
}  // namespace rpwa_amd

using namespace rpwa_amd;

extern "C" int rpwa_lik_hessian(rpwa_lik_ctx* ctx, const double* prodAmps, uint32_t nmbProdAmps,
                                double prodAmpFlat, uint32_t rank, double* hessian, double* flatTerms,
                                double* hessianFlat)
{
	clear_error();
	if (!ctx) {
		set_error("rpwa_lik_hessian: null context");
		return RPWA_ERR_INVALID;
	}
	if (!ctx->loaded) {
		set_error("rpwa_lik_hessian: decay amplitudes not loaded");
		return RPWA_ERR_STATE;
	}
	if (!prodAmps || !hessian || !flatTerms || !hessianFlat || rank == 0) {
		set_error("rpwa_lik_hessian: null output or rank 0");
		return RPWA_ERR_INVALID;
	}
	const AmpLayout& lay = ctx->lay;
	const uint32_t wmax = lay.wmax;
	if ((uint64_t)nmbProdAmps != (uint64_t)rank * 2 * wmax) {
		set_error("rpwa_lik_hessian: nmbProdAmps must be rank*2*nmbWavesMax");
		return RPWA_ERR_INVALID;
	}
	try {
		RPWA_HIP_CHECK(hipSetDevice(ctx->device));
		const bool mixed = lay.precision == RPWA_PREC_MIXED;
		// complex columns of the rows d and A (with the sectors' padding, whose columns are zero)
		const uint32_t cD = rank * lay.rowLen, cA = lay.rowLen;
		const uint32_t nTD = (2 * cD + 15) / 16, nTA = (2 * cA + 15) / 16;
		const size_t tD = (size_t)nTD * (nTD + 1) / 2, tA = (size_t)nTA * (nTA + 1) / 2;
		const size_t nWg = (size_t)std::max(ctx->nCu, 1);
		// event chunk: S and the weights within about 8 GiB
		const uint64_t chunk = std::max<uint64_t>(1024, (8ull << 30) / (32ull * rank + 16));
		const uint64_t cn = std::min<uint64_t>(chunk, lay.nEvents);
		if (ctx->device < 0 || ctx->device >= kHessDevices) {
			set_error("rpwa_lik_hessian: device index out of range");
			return RPWA_ERR_INVALID;
		}
		// one allocation: S [cn][2 rank], weights wD, wA [cn], T [rank][rowLen], the
		// workgroups' tiles, column and weight sums, and their reduction
		const size_t nCol = 16 * (size_t)nTD;  // column sums: [8 nTD] complex
		const size_t offWD = align256(cn * 2 * rank * sizeof(double2));
		const size_t offWA = offWD + align256(cn * sizeof(double));
		const size_t offT = offWA + align256(cn * sizeof(double));
		const size_t offPD = offT + align256((size_t)cD * sizeof(double2));
		const size_t offPA = offPD + align256(nWg * tD * 256 * sizeof(double));
		const size_t offCol = offPA + align256(nWg * tA * 256 * sizeof(double));
		const size_t offW = offCol + align256(nWg * nCol * sizeof(double));
		const size_t nRed = (tD + tA) * 256 + nCol;
		const size_t offRed = offW + align256(2 * nWg * sizeof(double));
		const size_t need = offRed + align256(nRed * sizeof(double));
		HessWork& work = hess_work(ctx->device);
		std::lock_guard<std::mutex> lock(work.m);
		if (need > work.cap) {
			(void)hipFree(work.buf);
			work.buf = nullptr;
			work.cap = 0;
			if (hipMalloc(&work.buf, need) != hipSuccess) {
				work.buf = nullptr;
				set_error("rpwa_lik_hessian: device allocation failed");
				return RPWA_ERR_NOMEM;
			}
			work.cap = need;
		}
		auto at = [&](size_t off) { return reinterpret_cast<double*>(work.buf + off); };
		hipStream_t s = nullptr;
		std::vector<double2> T(cD, make_double2(0., 0.));
		for (uint32_t r = 0; r < rank; ++r)
			for (uint32_t sec = 0; sec < 2; ++sec)
				std::memcpy(&T[(size_t)r * lay.rowLen + lay.secOff[sec]],
				            prodAmps + 2 * ((size_t)r * 2 + sec) * wmax, lay.nW[sec] * sizeof(double2));
		RPWA_HIP_CHECK(hipMemcpy(at(offT), T.data(), T.size() * sizeof(double2), hipMemcpyHostToDevice));
		std::vector<double> red(nRed), wsums(2 * nWg);
		const auto passes = mixed ? launch_hessian_passes_c64 : launch_hessian_passes_f64;
		hipError_t e = hipSuccess;
		for (uint64_t e0 = 0; e == hipSuccess && e0 < lay.nEvents; e0 += cn) {
			const uint64_t n = std::min<uint64_t>(cn, lay.nEvents - e0);
			const uint32_t nb = (uint32_t)std::min<uint64_t>((n + 63) / 64, 8ull * nWg);
			const bool narrow = lay.rowLen <= kNarrow;
			hipLaunchKernelGGL(mixed ? (narrow ? hessian_s_kernel<true, 4> : hessian_s_kernel<true, 16>)
			                         : (narrow ? hessian_s_kernel<false, 4> : hessian_s_kernel<false, 16>),
			                   dim3(nb), dim3(256), 0, s, ctx->d_amps, e0, n, lay.rowLen, lay.secOff[1], rank,
			                   reinterpret_cast<const double2*>(at(offT)), prodAmpFlat * prodAmpFlat,
			                   reinterpret_cast<double2*>(work.buf), at(offWD), at(offWA));
			e = hipGetLastError();
			hp::PassArgs a{};
			a.amps = ctx->d_amps;
			a.e0 = e0;
			a.n = n;
			a.rowLen = lay.rowLen;
			a.secOff1 = lay.secOff[1];
			a.rank2 = 2 * rank;
			a.S = reinterpret_cast<const double2*>(work.buf);
			a.accumulate = e0 > 0 ? 1 : 0;
			a.nCols = cD;
			a.nT = nTD;
			a.w = at(offWD);
			a.partials = at(offPD);
			a.nTiles = (uint32_t)tD;
			a.wsum = at(offW);
			a.colSum = reinterpret_cast<double2*>(at(offCol));
			if (e == hipSuccess)
				e = passes(true, a, (int)nWg, s);
			a.nCols = cA;
			a.nT = nTA;
			a.w = at(offWA);
			a.partials = at(offPA);
			a.nTiles = (uint32_t)tA;
			a.wsum = nullptr;
			if (e == hipSuccess)
				e = passes(false, a, (int)nWg, s);
		}
		double* const dRed = at(offRed);
		if (e == hipSuccess)
			e = launch_column_sum(at(offPD), (int)nWg, (uint32_t)(tD * 256), dRed, s);
		if (e == hipSuccess)
			e = launch_column_sum(at(offPA), (int)nWg, (uint32_t)(tA * 256), dRed + tD * 256, s);
		if (e == hipSuccess)
			e = launch_column_sum(at(offCol), (int)nWg, (uint32_t)nCol, dRed + (tD + tA) * 256, s);
		if (e == hipSuccess)
			e = hipMemcpyAsync(red.data(), dRed, nRed * sizeof(double), hipMemcpyDeviceToHost, s);
		if (e == hipSuccess)
			e = hipMemcpyAsync(wsums.data(), at(offW), 2 * nWg * sizeof(double), hipMemcpyDeviceToHost, s);
		if (e != hipSuccess)
			(void)hipStreamSynchronize(s);  // nothing of this call may still run on the work area
		RPWA_HIP_CHECK(e);
		RPWA_HIP_CHECK(hipStreamSynchronize(s));
		double f1 = 0., f2 = 0.;  // sums of factor and factor^2
		for (size_t g = 0; g < nWg; ++g) {
			f1 += wsums[2 * g];
			f2 += wsums[2 * g + 1];
		}
		const double* const tilesD = red.data();
		const double* const tilesA = tilesD + tD * 256;
		const double* const colD = tilesA + tA * 256;
		// assemble [rank][2][wmax] x [rank][2][wmax] x 3 (pwaLikelihood.cc:697-753)
		const size_t ndFull = (size_t)rank * 2 * wmax;
		std::vector<int> valid(ndFull, -1), gwave(ndFull, 0);  // columns of the rows d and A
		for (uint32_t r = 0; r < rank; ++r)
			for (uint32_t sec = 0; sec < 2; ++sec)
				for (uint32_t i = 0; i < lay.nW[sec]; ++i) {
					const size_t a = ((size_t)r * 2 + sec) * wmax + i;
					gwave[a] = (int)(lay.secOff[sec] + i);
					valid[a] = (int)(r * lay.rowLen) + gwave[a];
				}
		// row r of the symmetric matrix from its upper-triangle tiles (products of rows
		// with themselves: the halves of a diagonal tile are bitwise equal)
		auto matrix_row = [](const double* tiles, uint32_t nT, uint32_t r, double* out) {
			const uint32_t I = r / 16, i = r % 16;
			for (uint32_t J = 0; J < nT; ++J) {
				const uint32_t lo = std::min(I, J), hi = std::max(I, J);
				const double* t = tiles + ((size_t)lo * nT - (size_t)lo * (lo - 1) / 2 + (hi - lo)) * 256;
				for (uint32_t j = 0; j < 16; ++j)
					out[16 * J + j] = J < I ? t[16 * j + i] : t[16 * i + j];
			}
		};
		// sum of factor A_a conj(A_b) over the columns of a row: [cA][cA] real and imaginary parts
		std::vector<double> row0(16 * (size_t)std::max(nTD, nTA)), row1(row0.size());
		std::vector<double2> Q((size_t)cA * cA);
		for (uint32_t a = 0; a < cA; ++a) {
			matrix_row(tilesA, nTA, 2 * a, row0.data());
			matrix_row(tilesA, nTA, 2 * a + 1, row1.data());
			for (uint32_t b = 0; b < cA; ++b)
				Q[(size_t)a * cA + b] = make_double2(row0[2 * b] + row1[2 * b + 1], row1[2 * b] - row0[2 * b + 1]);
		}
		std::memset(hessian, 0, ndFull * ndFull * 3 * sizeof(double));
		for (size_t a = 0; a < ndFull; ++a) {
			const int va = valid[a];
			if (va < 0) {
				flatTerms[2 * a] = flatTerms[2 * a + 1] = 0.;
				continue;
			}
			const size_t blockA = a / wmax;  // (rank, sector)
			matrix_row(tilesD, nTD, 2 * va, row0.data());
			matrix_row(tilesD, nTD, 2 * va + 1, row1.data());
			for (size_t b = 0; b < ndFull; ++b) {
				const int vb = valid[b];
				if (vb < 0)
					continue;
				double* h = hessian + (a * ndFull + b) * 3;
				h[0] = row0[2 * vb];
				h[1] = row0[2 * vb + 1];
				h[2] = row1[2 * vb + 1];
				if (b / wmax == blockA) {
					const double2 q = Q[(size_t)gwave[a] * cA + gwave[b]];
					h[0] -= q.x;
					h[1] -= q.y;
					h[2] -= q.x;
				}
			}
			flatTerms[2 * a] = prodAmpFlat * colD[2 * va];
			flatTerms[2 * a + 1] = prodAmpFlat * colD[2 * va + 1];
		}
		*hessianFlat = prodAmpFlat * prodAmpFlat * f2 - f1;
		return RPWA_OK;
	} catch (const std::exception& ex) {
		set_error(std::string("rpwa_lik_hessian: ") + ex.what());
		return RPWA_ERR_NOMEM;
	}
}
