// hessian_pass.h -- rank-k passes of the Hessian (hessian.hip) over the windows, tiles
// and pairs of waves of rank_update.h, with rows that are formed here instead of
// copied: loads of a chunk's amplitudes and S are in flight beside the products of
// the chunk before it, the entries are stored to LDS between the later products.
// Bound by FP64 MFMA (64 cycles per tile and step) plus the vector work of forming
// the rows, which takes the same unit: 42 to 54 TFLOP/s at 28 to 66 tiles per pass; a
// pass with more tiles forms fewer entries per product.
#pragma once

#include <cstdint>
#include <type_traits>
#include <utility>

#include "rank_update.h"

namespace rpwa_amd {
namespace hp {

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

// all passes over the rows d (dRows) or A
template <bool MIXED>
hipError_t launch_passes(bool dRows, PassArgs a, int nWg, hipStream_t s)
{
	const uint32_t nWin = a.nT <= kOneWin ? 1 : (a.nT + kMaxWin - 1) / kMaxWin;
	double* const wsum = a.wsum;
	for (uint32_t u = 0; u < nWin; ++u)
		for (uint32_t v = u; v < nWin; ++v) {
			uint32_t nI, nJ;
			ru::window(a.nT, nWin, u, a.winI0, nI);
			ru::window(a.nT, nWin, v, a.winJ0, nJ);
			const int j = v > u ? (int)nJ : 0;
			const PassKernel p = dRows ? pick_pass<MIXED, true>((int)nI, j) : pick_pass<MIXED, false>((int)nI, j);
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

}  // namespace hp

// complex64 and complex128 amplitudes (hessian_pass_c64.hip, hessian_pass_f64.hip)
hipError_t launch_hessian_passes_c64(bool dRows, const hp::PassArgs& a, int nWg, hipStream_t s);
hipError_t launch_hessian_passes_f64(bool dRows, const hp::PassArgs& a, int nWg, hipStream_t s);

}  // namespace rpwa_amd
