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
// 2M events x 88 waves x rank 2, complex64 amplitudes: 9.98 -> 7.28 ms; before, a
// kernel wrote the rows (8.5 GB, 2.3 ms) and weighted passes read them (7.1 ms).
#include "event_kernel.h"
#include "rank_update.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

namespace rpwa_amd {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

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

// ---------------------------------------------------------------------------
// Rank-k passes over the windows, tiles and pairs of waves of rank_update.h, with
// rows that are formed here instead of copied: loads of a chunk's amplitudes and S
// are in flight beside the products of the chunk before it, the entries are stored
// to LDS between the later products.  Bound by FP64 MFMA (64 cycles per tile and
// step) plus the vector work of forming the rows, which takes the same unit: 41 to
// 53 TFLOP/s at 28 to 66 tiles per pass; a pass with more tiles forms fewer entries
// per product.
using ru::d4;
using ru::kLdsBytes;
using ru::kThreads;
// one window up to 11 blocks: a 12-block triangle's sums and staged loads do not fit
// the registers of a wave
constexpr int kOneWin = 11, kMaxWin = ru::kMaxWin;

// LDS image of a pass
template <int NI, int NJ>
struct Pass : ru::Tiles<NI, NJ> {
	typedef ru::Tiles<NI, NJ> Base;
	using Base::NB;
	using Base::most;
	using Base::rect;
	static constexpr int NC = 8 * NB;                 // complex columns staged
	static constexpr int PER = kThreads / NC;         // events staged per step
	static constexpr int STRIDE = 16 * NB + 1;        // doubles per LDS row: odd
	static constexpr int chFit = kLdsBytes / (2 * 8 * STRIDE) / 8 * 8;
	static constexpr int CH = chFit < 64 ? chFit : 64;  // events per chunk
	static constexpr int BUF = CH * STRIDE;
	static constexpr int steps = (CH + PER - 1) / PER;
	// operands read a step ahead where the registers hold two sets beside the sums
	static constexpr int ahead = rect ? 1 : 0;
	// both buffers, and after the hand-over the threads' column and factor sums
	static constexpr size_t lds = (2 * BUF > 4 * kThreads ? 2 * (size_t)BUF : 4 * (size_t)kThreads) * sizeof(double);
	// staging steps whose loads are in flight together: what the 256 registers leave
	// beside the sums and operands, all of a chunk's where they fit (measured for the
	// d triangles, whose column sums take more)
	static constexpr int batch(bool mixed, bool dRows)
	{
		if (dRows && !rect)
			return steps < 4 ? steps : 4;
		const int perStep = (mixed ? 2 : 4) + (dRows ? 4 : 2);
		const int fit = (200 - 8 * most - 4 * NB) / perStep;
		return fit < 2 ? 2 : fit < steps ? fit : steps;
	}
	static_assert(2 * BUF >= 4 * most * 256, "the waves' sums are handed over in one round");
};

struct PassArgs {
	const void* amps;      // [events][rowLen] complex
	uint64_t e0, n;        // events of this call
	uint32_t rowLen, secOff1, rank2;
	uint32_t nCols;        // complex columns of a row: rank rowLen (d) or rowLen (A)
	uint32_t nT;           // column blocks of a row
	uint32_t winI0, winJ0; // first block of the windows
	const double2* S;      // [n][2 rank], times factor (d rows)
	const double* w;       // [n] factor (d rows) or its square root (A rows)
	double* partials;      // [nWg][tiles of the triangle][256]
	uint32_t nTiles;
	double* wsum;          // [nWg][2] sums of factor and factor^2, by the first pass over d; null in the others
	double2* colSum;       // [nWg][8 nT]: sum of factor^2 d, by the triangle passes
	int accumulate;        // later calls of a long event list add to the partials
};

// operands of a wave's 4-event step: the column blocks its tiles use
template <class P, int G>
__device__ __forceinline__ void pass_read(const double* __restrict__ xr, double (&v)[P::NB])
{
	constexpr uint32_t used = P::blocks(G, false);
#pragma unroll
	for (int b = 0; b < P::NB; ++b)
		v[b] = (used >> b & 1) ? xr[16 * b] : 0.;
}

template <class P, int G, int... Q>
__device__ __forceinline__ void pass_step(const double (&v)[P::NB], d4* acc, std::integer_sequence<int, Q...>)
{
	constexpr int t0 = P::begin(G);
	((acc[Q] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[ru::TileRC<P, t0 + Q>::r], v[ru::TileRC<P, t0 + Q>::c], acc[Q], 0, 0, 0)),
	 ...);
}

template <bool MIXED, bool DROWS, class P, int G>
__device__ __forceinline__ void pass_body(const PassArgs& a, double* lds, double2* csh, double2* wsh)
{
	constexpr int NG = P::size(G);
	constexpr int kBatch = P::batch(MIXED, DROWS), kBatches = (P::steps + kBatch - 1) / kBatch;
	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int h = tid >> 8;  // which wave of the pair (waves 0-3 or 4-7)
	const int li = lane & 15, lk = lane >> 4;

	d4 acc[NG > 0 ? NG : 1];
#pragma unroll
	for (int q = 0; q < NG; ++q)
		acc[q] = d4{0., 0., 0., 0.};

	// a thread stages one complex column k of the windows, for the events sEv, sEv +
	// PER, ... of a chunk; columns past the row (the last window's padding) are zeros
	const uint32_t k = tid % P::NC, sEv = tid / P::NC;
	const uint32_t col = k < 8u * P::nI ? 8 * a.winI0 + k : 8 * a.winJ0 + (k - 8 * P::nI);
	const bool stager = sEv < (uint32_t)P::PER, valid = stager && col < a.nCols;
	const uint32_t rank = DROWS && valid ? col / a.rowLen : 0;
	const uint32_t pos = valid ? col - rank * a.rowLen : 0;
	const uint32_t rs = 2 * rank + (pos >= a.secOff1 ? 1 : 0);
	double2 colAcc = make_double2(0., 0.);
	double2 wacc = make_double2(0., 0.);
	for (int i = tid; i < 2 * P::BUF; i += kThreads)
		lds[i] = 0.;
	__syncthreads();

	typedef typename std::conditional<MIXED, float2, double2>::type stored;
	const uint32_t rowBytes = a.rowLen * (uint32_t)sizeof(stored), sBytes = a.rank2 * 16;
	const uint32_t offA = sEv * rowBytes + pos * (uint32_t)sizeof(stored), offS = sEv * sBytes + rs * 16, offW = sEv * 8;
	stored ax[kBatch];
	double2 sx[kBatch];
	double wx[kBatch];
	// staging step st of chunk c into register set i: issue the loads ...
	auto loadStep = [&](uint64_t c, int st, int i) {
		const uint64_t first = c * P::CH;
		if (first + P::CH <= a.n) {  // a whole chunk: fixed offsets from a common base
			if (valid && (st * P::PER + P::PER <= P::CH || sEv + st * P::PER < (uint32_t)P::CH)) {
				const uint64_t e = first + (uint32_t)(st * P::PER);
				ax[i] = *reinterpret_cast<const stored*>(reinterpret_cast<const char*>(a.amps) + (a.e0 + e) * rowBytes + offA);
				if (DROWS)
					sx[i] = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(a.S) + e * sBytes + offS);
				if (!DROWS || !P::rect)
					wx[i] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(a.w + e) + offW);
			}
		} else if (valid) {  // the last chunk: past the list's end the last event, dropped below
			const uint64_t e = min(first + sEv + (uint32_t)(st * P::PER), a.n - 1);
			ax[i] = reinterpret_cast<const stored*>(a.amps)[(a.e0 + e) * a.rowLen + pos];
			if (DROWS)
				sx[i] = a.S[e * a.rank2 + rs];
			if (!DROWS || !P::rect)
				wx[i] = a.w[e];
		}
	};
	// ... and form the row entries and store them
	auto storeStep = [&](uint64_t c, int st, int i, double* xs) {
		const uint32_t e = sEv + (uint32_t)(st * P::PER);
		if (valid && (st * P::PER + P::PER <= P::CH || e < (uint32_t)P::CH)) {
			double2 x = make_double2((double)ax[i].x, (double)ax[i].y);
			if (DROWS)  // d = S conj(A)
				x = make_double2(sx[i].x * x.x + sx[i].y * x.y, sx[i].y * x.x - sx[i].x * x.y);
			else
				x = make_double2(wx[i] * x.x, wx[i] * x.y);
			if ((c + 1) * P::CH > a.n && c * P::CH + e >= a.n)
				x = make_double2(0., 0.);
			xs[e * P::STRIDE + 2 * k] = x.x;
			xs[e * P::STRIDE + 2 * k + 1] = x.y;
			if (DROWS && !P::rect) {
				colAcc.x = fma(wx[i], x.x, colAcc.x);
				colAcc.y = fma(wx[i], x.y, colAcc.y);
				if (k == 0 && a.wsum && c * P::CH + e < a.n) {
					wacc.x += wx[i];
					wacc.y = fma(wx[i], wx[i], wacc.y);
				}
			}
		}
	};
	const uint64_t nChunks = (a.n + P::CH - 1) / P::CH;
	uint64_t c = blockIdx.x;
	int buf = 0;
	if (c < nChunks) {
#pragma unroll
		for (int s0 = 0; s0 < P::steps; s0 += kBatch) {
#pragma unroll
			for (int i = 0; i < kBatch && s0 + i < P::steps; ++i)
				loadStep(c, s0 + i, i);
#pragma unroll
			for (int i = 0; i < kBatch && s0 + i < P::steps; ++i)
				storeStep(c, s0 + i, i, lds);
		}
	}
	__syncthreads();
	constexpr int KK = P::CH / 8;
	for (; c < nChunks; c += gridDim.x) {
		const uint64_t next = c + gridDim.x;
		const bool more = next < nChunks;
		const double* xs = lds + buf * P::BUF;
		double* xn = lds + (buf ^ 1) * P::BUF;
		// products 8 events at a time (4 per wave), in the rectangles with operands a step
		// ahead (the two waves of a SIMD issue in turn and would wait for their reads
		// together); the steps of a batch are loaded in front of the batch's share of the
		// products and stored one by one during its second half
		double v[1 + P::ahead][P::NB];
		if (P::ahead)
			pass_read<P, G>(xs + (h * 4 + lk) * P::STRIDE + li, v[0]);
#pragma unroll
		for (int part = 0; part < kBatches; ++part) {
			const int s0 = part * kBatch, s1 = s0 + kBatch < P::steps ? s0 + kBatch : P::steps;
			const int k0 = part * KK / kBatches, k1 = (part + 1) * KK / kBatches;
			const int kMid = k0 + (k1 - k0) / 2;
			if (more) {
#pragma unroll
				for (int st = s0; st < s1; ++st)
					loadStep(next, st, st - s0);
			}
#pragma unroll
			for (int kk = k0; kk < k1; ++kk) {
				if (P::ahead ? kk + 1 < KK : true)
					pass_read<P, G>(xs + ((2 * (kk + P::ahead) + h) * 4 + lk) * P::STRIDE + li, v[(kk + P::ahead) & P::ahead]);
				__builtin_amdgcn_sched_barrier(0);
				pass_step<P, G>(v[kk & P::ahead], acc, std::make_integer_sequence<int, NG>{});
				__builtin_amdgcn_sched_barrier(0);
				if (more && kk >= kMid) {
#pragma unroll
					for (int st = s0 + (s1 - s0) * (kk - kMid) / (k1 - kMid); st < s0 + (s1 - s0) * (kk + 1 - kMid) / (k1 - kMid); ++st)
						storeStep(next, st, st - s0, xn);
				}
				__builtin_amdgcn_sched_barrier(0);
			}
		}
		__syncthreads();
		buf ^= 1;
	}

	// the second wave of a pair hands its sums to the first; v_mfma_f64_16x16x4_f64
	// leaves D[i][j] in lane j + 16 (i % 4), register i / 4.  Tiles past the row are dropped
	double* red = lds + G * P::most * 256;
	double* out = a.partials + (size_t)blockIdx.x * a.nTiles * 256;
	if (h == 1) {
#pragma unroll
		for (int q = 0; q < NG; ++q)
#pragma unroll
			for (int v = 0; v < 4; ++v)
				red[(q * 4 + v) * 64 + lane] = acc[q][v];
	}
	__syncthreads();
	if (h == 0) {
#pragma unroll
		for (int q = 0; q < NG; ++q) {
			const int at = P::place(P::begin(G) + q, a.winI0, a.winJ0, a.nT);
			if (at < 0)
				continue;
			double* o = out + (size_t)at * 256;
#pragma unroll
			for (int v = 0; v < 4; ++v)
				acc[q][v] += red[(q * 4 + v) * 64 + lane];
			if (a.accumulate) {
#pragma unroll
				for (int v = 0; v < 4; ++v)
					acc[q][v] += o[(lk + 4 * v) * 16 + li];
			}
#pragma unroll
			for (int v = 0; v < 4; ++v)
				o[(lk + 4 * v) * 16 + li] = acc[q][v];
		}
	}
	__syncthreads();  // the hand-over has been read: its area takes the column and weight sums
	csh[tid] = colAcc;
	wsh[tid] = wacc;
	__syncthreads();
	if (DROWS && !P::rect && tid < P::NC && col < 8 * a.nT) {
		double2 s = make_double2(0., 0.);
		for (int p = 0; p < P::PER; ++p) {
			s.x += csh[p * P::NC + tid].x;
			s.y += csh[p * P::NC + tid].y;
		}
		double2* o = a.colSum + (size_t)blockIdx.x * (8 * a.nT) + col;
		if (a.accumulate) {
			s.x += o->x;
			s.y += o->y;
		}
		*o = s;
	}
	if (DROWS && a.wsum && tid == 0) {
		double2 s = make_double2(0., 0.);
		for (int r = 0; r < P::PER * P::NC; r += P::NC) {  // the threads of column 0
			s.x += wsh[r].x;
			s.y += wsh[r].y;
		}
		double* o = a.wsum + 2 * blockIdx.x;
		o[0] = a.accumulate ? o[0] + s.x : s.x;
		o[1] = a.accumulate ? o[1] + s.y : s.y;
	}
}

template <bool MIXED, bool DROWS, int NI, int NJ>
__global__ __launch_bounds__(kThreads) void hessian_pass_kernel(PassArgs a)
{
	typedef Pass<NI, NJ> P;
	extern __shared__ double lds[];
	double2* csh = reinterpret_cast<double2*>(lds);  // after the hand-over (barriers between)
	double2* wsh = csh + kThreads;
	// wave-uniform branch: waves g and g + 4 run group g
	switch ((threadIdx.x >> 6) & 3) {
	case 0: pass_body<MIXED, DROWS, P, 0>(a, lds, csh, wsh); break;
	case 1: pass_body<MIXED, DROWS, P, 1>(a, lds, csh, wsh); break;
	case 2: pass_body<MIXED, DROWS, P, 2>(a, lds, csh, wsh); break;
	default: pass_body<MIXED, DROWS, P, 3>(a, lds, csh, wsh); break;
	}
}

struct PassKernel {
	void (*k)(PassArgs) = nullptr;
	size_t lds = 0;
};

template <bool MIXED, bool DROWS, int NI, int NJ>
PassKernel make_pass()
{
	return PassKernel{hessian_pass_kernel<MIXED, DROWS, NI, NJ>, Pass<NI, NJ>::lds};
}

// windows of nI and nJ blocks (nJ = 0: the triangle); nJ is nI or one less
template <bool MIXED, bool DROWS>
PassKernel pick_pass(int nI, int nJ)
{
	switch (nI * 16 + nJ) {
	case 0x10: return make_pass<MIXED, DROWS, 1, 0>();
	case 0x20: return make_pass<MIXED, DROWS, 2, 0>();
	case 0x30: return make_pass<MIXED, DROWS, 3, 0>();
	case 0x40: return make_pass<MIXED, DROWS, 4, 0>();
	case 0x50: return make_pass<MIXED, DROWS, 5, 0>();
	case 0x60: return make_pass<MIXED, DROWS, 6, 0>();
	case 0x70: return make_pass<MIXED, DROWS, 7, 0>();
	case 0x80: return make_pass<MIXED, DROWS, 8, 0>();
	case 0x90: return make_pass<MIXED, DROWS, 9, 0>();
	case 0xA0: return make_pass<MIXED, DROWS, 10, 0>();
	case 0xB0: return make_pass<MIXED, DROWS, 11, 0>();
	case 0x65: return make_pass<MIXED, DROWS, 6, 5>();
	case 0x66: return make_pass<MIXED, DROWS, 6, 6>();
	case 0x76: return make_pass<MIXED, DROWS, 7, 6>();
	case 0x77: return make_pass<MIXED, DROWS, 7, 7>();
	case 0x87: return make_pass<MIXED, DROWS, 8, 7>();
	case 0x88: return make_pass<MIXED, DROWS, 8, 8>();
	default: return PassKernel();
	}
}

hipError_t launch_passes(bool mixed, bool dRows, PassArgs a, int nWg, hipStream_t s)
{
	const uint32_t nWin = a.nT <= kOneWin ? 1 : (a.nT + kMaxWin - 1) / kMaxWin;
	double* const wsum = a.wsum;
	for (uint32_t u = 0; u < nWin; ++u)
		for (uint32_t v = u; v < nWin; ++v) {
			uint32_t nI, nJ;
			ru::window(a.nT, nWin, u, a.winI0, nI);
			ru::window(a.nT, nWin, v, a.winJ0, nJ);
			const int j = v > u ? (int)nJ : 0;
			const PassKernel p = mixed ? (dRows ? pick_pass<true, true>((int)nI, j) : pick_pass<true, false>((int)nI, j))
			                           : (dRows ? pick_pass<false, true>((int)nI, j) : pick_pass<false, false>((int)nI, j));
			if (!p.k)
				return hipErrorInvalidValue;
			a.wsum = u == 0 && v == 0 ? wsum : nullptr;
			if (p.lds > 64u * 1024u)
				if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(p.k),
				                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds))
					return e;
			hipLaunchKernelGGL(p.k, dim3(nWg), dim3(kThreads), p.lds, s, a);
			if (hipError_t e = hipGetLastError())
				return e;
		}
	return hipSuccess;
}

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
			PassArgs a{};
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
				e = launch_passes(mixed, true, a, (int)nWg, s);
			a.nCols = cA;
			a.nT = nTA;
			a.w = at(offWA);
			a.partials = at(offPA);
			a.nTiles = (uint32_t)tA;
			a.wsum = nullptr;
			if (e == hipSuccess)
				e = launch_passes(mixed, false, a, (int)nWg, s);
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
