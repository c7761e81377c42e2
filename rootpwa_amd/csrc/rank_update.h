// rank_update.h -- rank-k updates sum_e w_e x_e x_e^T of real event rows on
// v_mfma_f64_16x16x4_f64 (the normalisation integral and the Hessian).
//
// A row of D doubles is cut into column blocks of 16; the output is the tiles
// (16 x 16) of the upper triangle of blocks.  Rows of up to kOneWin blocks are one
// window, wider ones are cut into windows of at most kMaxWin blocks of nearly
// equal size; a pass computes the tiles of a window's triangle (NJ = 0) or
// between two windows (NI x NJ), so that every tile is computed by exactly one
// pass.  One workgroup of 8 waves per CU walks chunks of CH events, two of them in
// LDS.  The tiles are split over four pairs of waves {g, g + 4} (one SIMD each) at
// compile time; the waves of a pair take alternate 4-event steps, each reading the
// operand blocks of its tiles once per step, one step ahead.
//
// Bound by FP64 MFMA (64 cycles per tile and step).  What slows it down is other
// vector instructions: one of another wave of the SIMD waits for a whole FP64
// MFMA.  A copy of a chunk's rows through registers (loads, addresses, LDS stores)
// adds to the products instead of running beside them (5M events x 88 waves:
// products alone 2.3 ms, copy alone 1.3 ms, both 2.7 to 3.4 ms), so a chunk is
// copied by global_load_lds, whose addresses are a scalar base and lane offsets
// that stay the same for every chunk: a call 2.73 -> 2.59 ms (65 TFLOP/s of issued
// products).  Weights cost FP64 multiplies of the operands (2M x 88: 1.05 -> 1.11 ms).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <utility>

namespace rpwa_amd {
namespace ru {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kOneWin = 12, kMaxWin = 8;
constexpr int kLdsBytes = 160 * 1024;

constexpr int tri_row(int n, int t)
{
	int i = 0;
	while (t >= n - i) {
		t -= n - i;
		++i;
	}
	return i;
}
constexpr int tri_col(int n, int t)
{
	const int i = tri_row(n, t);
	return t - (i * n - i * (i - 1) / 2) + i;
}

// the tiles of a pass over windows of NI and NJ blocks and their split over the four
// pairs of waves
template <int NI, int NJ>
struct Tiles {
	static constexpr bool rect = NJ > 0;
	static constexpr int nI = NI;
	static constexpr int NB = NI + NJ;  // column blocks in LDS
	static constexpr int tiles = rect ? NI * NJ : NI * (NI + 1) / 2;
	static constexpr int nJ = rect ? NJ : 1;
	static constexpr int row(int t) { return rect ? t / nJ : tri_row(NI, t); }
	static constexpr int col(int t) { return rect ? NI + t % nJ : tri_col(NI, t); }
	static constexpr int begin(int g) { return g * tiles / 4; }
	static constexpr int size(int g) { return begin(g + 1) - begin(g); }
	static constexpr int most = (tiles + 3) / 4;
	// the column blocks that group g reads (rowsOnly: as the left operand)
	static constexpr uint32_t blocks(int g, bool rowsOnly)
	{
		uint32_t m = 0;
		for (int t = begin(g); t < begin(g + 1); ++t)
			m |= 1u << row(t) | (rowsOnly ? 0u : 1u << col(t));
		return m;
	}
	// place of tile t in a row of nT blocks' triangle, or -1 past the row
	static __device__ __forceinline__ int place(int t, uint32_t winI0, uint32_t winJ0, uint32_t nT)
	{
		if (!rect && NI > kMaxWin)  // the only window
			return t;
		const uint32_t I = winI0 + row(t), J = rect ? winJ0 + (col(t) - NI) : winI0 + col(t);
		return J < nT ? (int)(I * nT - I * (I - 1) / 2 + (J - I)) : -1;
	}
};

// LDS image of a pass that copies its rows
template <int NI, int NJ>
struct Pass : Tiles<NI, NJ> {
	typedef Tiles<NI, NJ> Base;
	using Base::NB;
	using Base::most;
	static constexpr int ROW = 16 * NB;    // doubles per LDS row
	static constexpr int UNITS = 8 * NB;   // 16-byte units per LDS row
	// events per chunk: the largest multiple of 8 (a step of both waves of a pair) up
	// to 64 whose two buffers, rows and weights, fit LDS (56 for 11 blocks)
	static constexpr int fit = (kLdsBytes - 1024) / (2 * 8 * (ROW + 1)) / 8 * 8;
	static constexpr int CH = fit < 64 ? fit : 64;
	static constexpr int LOADS = (CH * UNITS + kThreads - 1) / kThreads;  // copies per wave and chunk, of 64 units
	static_assert(CH * UNITS % 64 == 0, "copies of whole waves");
	static constexpr int bufDoubles = CH * ROW;
	// the rows of both buffers and their weights; afterwards the waves' sums in rounds
	// of ROUND tiles per group
	static constexpr int doubles = 2 * bufDoubles + 2 * CH;
	static constexpr int ROUND = doubles / (4 * 256) < most ? doubles / (4 * 256) : most;
	static constexpr size_t lds = doubles * sizeof(double);
	// Rows whose length is a multiple of 32 doubles start in the same bank: there odd
	// rows have neighbouring blocks exchanged, so that the four rows of an operand
	// read use all banks
	static constexpr uint32_t flip = NB % 2 == 0 ? 1 : 0;
};

struct Args {
	const double* x;        // [n][D]
	const double* w;        // weights or null
	uint64_t n;
	uint32_t D;             // doubles per row (even)
	uint32_t nT;            // column blocks of a row
	uint32_t winI0, winJ0;  // first block of the windows
	uint32_t nTiles;        // tiles of the triangle
	double* partials;       // [nWg][nTiles][256]
	double* wsum;           // [nWg] sums of the weights, by the first pass; null in the others
	int accumulate;         // add to the partials of an earlier call
	int direct;             // weight w[e] instead of 1 / w[e]
	int odd;                // x is not 16-byte aligned (set by launch)
};

// 16 bytes per lane of global memory straight into LDS: lane l of the wave
// writes base + 16 l.  In assembly because the compiler would let every later
// LDS read wait for it; there is no register result, and the waits are explicit
__device__ __forceinline__ void copy16(const double* base, uint32_t off, uint32_t ldsBase)
{
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(ldsBase), "v"(off), "s"(base)
	             : "memory", "m0");
}

// 4 bytes per lane, for rows that are not 16-byte aligned: lane l writes base + 4 l
__device__ __forceinline__ void copy4(const double* base, uint32_t off, uint32_t ldsBase)
{
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(ldsBase), "v"(off), "s"(base)
	             : "memory", "m0");
}

template <class P, int T>
struct TileRC {
	static constexpr int r = P::row(T), c = P::col(T);
};

// operands of a 4-event step: the column blocks the group's tiles use; xe, xo: the
// lane's place in the row for even and for odd blocks
template <class P, int G>
__device__ __forceinline__ void read_step(const double* __restrict__ xe, const double* __restrict__ xo, double (&v)[P::NB])
{
	constexpr uint32_t used = P::blocks(G, false);
#pragma unroll
	for (int b = 0; b < P::NB; ++b)
		v[b] = (used >> b & 1) ? (b & 1 ? xo : xe)[16 * b] : 0.;
}

template <class P, int G, bool WT, int... Q>
__device__ __forceinline__ void mfma_step(const double (&v)[P::NB], double wt, d4* acc,
                                          std::integer_sequence<int, Q...>)
{
	constexpr int t0 = P::begin(G);
	constexpr uint32_t rows = P::blocks(G, true);
	double va[P::NB];
#pragma unroll
	for (int b = 0; b < P::NB; ++b)
		va[b] = WT && (rows >> b & 1) ? v[b] * wt : v[b];
	((acc[Q] = __builtin_amdgcn_mfma_f64_16x16x4f64(va[TileRC<P, t0 + Q>::r], v[TileRC<P, t0 + Q>::c], acc[Q], 0, 0, 0)),
	 ...);
}

template <class P, bool WT, int G>
__device__ __forceinline__ void body(const Args& a, double* lds, double* wsh)
{
	constexpr int NG = P::size(G);
	constexpr int CH = P::CH;
	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int h = wave >> 2;  // which wave of the pair
	const int li = lane & 15, lk = lane >> 4;
	const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) double*)lds;
	double* const wts = lds + 2 * P::bufDoubles;  // [2][CH]

	d4 acc[NG > 0 ? NG : 1];
#pragma unroll
	for (int q = 0; q < NG; ++q)
		acc[q] = d4{0., 0., 0., 0.};

	// the unit a lane copies: number lane + 64 (wave + 8 i) of the chunk's LDS image;
	// past the row (the last window's padding) the row's last unit, whose products
	// only reach output elements past the row
	auto offset = [&](uint32_t u) {
		const uint32_t e = u / P::UNITS, p = (u % P::UNITS) ^ (P::flip * 8 * (e & 1));
		const uint32_t c = p < 8u * P::nI ? 8 * a.winI0 + p : 8 * a.winJ0 + (p - 8 * P::nI);
		return e * a.D * 8 + 16 * min(c, a.D / 2 - 1);
	};
	uint32_t off[P::LOADS];
#pragma unroll
	for (int i = 0; i < P::LOADS; ++i)
		off[i] = offset((uint32_t)(lane + 64 * (wave + kWaves * i)));
	// wave-uniform, and all but the last copy for every wave
	auto copies = [&](int i) {
		return 64 * (kWaves - 1 + kWaves * i) < CH * P::UNITS || 64 * (wave + kWaves * i) < CH * P::UNITS;
	};
	auto copy = [&](uint64_t c, int buf) {
		const double* base = a.x + c * CH * a.D;
		const uint32_t at = lds0 + buf * P::bufDoubles * 8;
		if (a.odd) {  // 16 units at a time, past the list's end its last unit
			const uint32_t last = (uint32_t)min(a.n - c * CH, (uint64_t)CH) * a.D * 8 - 16;
#pragma unroll 1
			for (int i = wave; i < CH * P::UNITS / 16; i += kWaves)
				copy4(base, min(offset(16 * i + lane / 4), last) + 4 * (lane % 4), at + 256 * i);
		} else if ((c + 1) * CH <= a.n) {
#pragma unroll
			for (int i = 0; i < P::LOADS; ++i)
				if (copies(i))
					copy16(base, off[i], at + 1024 * (wave + kWaves * i));
		} else {  // the last chunk: past the list's end its last unit, zeroed afterwards
			const uint32_t last = (uint32_t)(a.n - c * CH) * a.D * 8 - 16;
#pragma unroll
			for (int i = 0; i < P::LOADS; ++i)
				if (copies(i))
					copy16(base, min(off[i], last), at + 1024 * (wave + kWaves * i));
		}
	};
	// a weight is used where it is stored, after the products: an earlier use would
	// wait for the copies in flight as well
	double wacc = 0., wstage = 0.;
	auto loadWeight = [&](uint64_t c) {
		if (WT && tid < CH)
			wstage = a.w[min(c * CH + tid, a.n - 1)];
	};
	auto storeWeight = [&](uint64_t c, int buf) {
		if (WT && tid < CH) {
			const double w = c * CH + tid < a.n ? (a.direct ? wstage : 1. / wstage) : 0.;
			wts[buf * CH + tid] = w;
			wacc += w;
		}
	};
	// the chunk is in LDS (its copies of all waves have arrived)
	auto arrive = [&](uint64_t c, int buf) {
		asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
		__syncthreads();
		if ((c + 1) * CH > a.n) {  // rows past the list's end
			const int first = (int)(a.n - c * CH) * P::ROW;
			for (int i = first + tid; i < P::bufDoubles; i += kThreads)
				lds[buf * P::bufDoubles + i] = 0.;
			__syncthreads();
		}
	};

	const uint64_t nChunks = (a.n + CH - 1) / CH;
	uint64_t c = blockIdx.x;
	int buf = 0;
	if (c < nChunks) {
		loadWeight(c);
		copy(c, 0);
		storeWeight(c, 0);
		arrive(c, 0);
	}
	for (; c < nChunks; c += gridDim.x) {
		const uint64_t next = c + gridDim.x;
		if (next < nChunks) {
			loadWeight(next);
			copy(next, buf ^ 1);
		}
		const double* xr = lds + buf * P::bufDoubles + (4 * h + lk) * P::ROW + li;
		const int odd = P::flip * (lk & 1);
		const double *xe = xr + 16 * odd, *xo = xr - 16 * odd;
		if constexpr (WT) {
			// the multiplies take the matrix core's turns: with the operands a step ahead
			// they come in front of every step's products and wait there for the other
			// wave's (1M events x 64 waves: 420 us, in this order 380, unweighted 330)
#pragma unroll 1
			for (int s = 0; s < CH / 8; ++s) {
				double v[P::NB];
				read_step<P, G>(xe + s * 8 * P::ROW, xo + s * 8 * P::ROW, v);
				mfma_step<P, G, true>(v, wts[buf * CH + 4 * h + lk + 8 * s], acc, std::make_integer_sequence<int, NG>{});
			}
		} else {
			double v[2][P::NB];
			read_step<P, G>(xe, xo, v[0]);
			// steps 2 s + h, operands one step ahead; past the chunk the last is read again
#pragma unroll 1
			for (int s = 0; s < CH / 8; s += 2) {
				const int s1 = s + 1 < CH / 8 ? s + 1 : s, s2 = s + 2 < CH / 8 ? s + 2 : s;
				read_step<P, G>(xe + s1 * 8 * P::ROW, xo + s1 * 8 * P::ROW, v[1]);
				__builtin_amdgcn_sched_barrier(0);
				mfma_step<P, G, false>(v[0], 1., acc, std::make_integer_sequence<int, NG>{});
				__builtin_amdgcn_sched_barrier(0);
				if (s + 1 < CH / 8) {
					read_step<P, G>(xe + s2 * 8 * P::ROW, xo + s2 * 8 * P::ROW, v[0]);
					__builtin_amdgcn_sched_barrier(0);
					mfma_step<P, G, false>(v[1], 1., acc, std::make_integer_sequence<int, NG>{});
					__builtin_amdgcn_sched_barrier(0);
				}
			}
		}
		if (next < nChunks) {
			storeWeight(next, buf ^ 1);
			arrive(next, buf ^ 1);
		} else {
			__syncthreads();  // LDS is free for the hand-over
		}
		buf ^= 1;
	}

	// hand-over: the second wave of a pair passes its sums to the first through LDS in
	// rounds that every wave runs, and the first writes the pair's sum; tiles past the
	// row are dropped.  v_mfma_f64_16x16x4_f64 leaves D[i][j] in lane j + 16 (i % 4),
	// register i / 4.  Few branches and little address work a tile: short event lists
	// are bound by fetching this code (3000 events x 88 waves: 64 -> 56 us a call)
	double* red = lds + G * P::ROUND * 256;
	double* out = a.partials + (size_t)blockIdx.x * a.nTiles * 256;
#pragma unroll
	for (int r0 = 0; r0 < P::most; r0 += P::ROUND) {
		if (h == 1) {
#pragma unroll
			for (int q = r0; q < NG && q < r0 + P::ROUND; ++q)
#pragma unroll
				for (int v = 0; v < 4; ++v)
					red[((q - r0) * 4 + v) * 64 + lane] = acc[q][v];
		}
		__syncthreads();
		if (h == 0) {
#pragma unroll
			for (int q = r0; q < NG && q < r0 + P::ROUND; ++q) {
				const int at0 = P::place(P::begin(G) + q, a.winI0, a.winJ0, a.nT);
				if (at0 < 0)
					continue;
				double* o = out + (size_t)at0 * 256;
#pragma unroll
				for (int v = 0; v < 4; ++v)
					acc[q][v] += red[((q - r0) * 4 + v) * 64 + lane];
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
		__syncthreads();
	}
	if (WT) {
		if (tid < CH)
			wsh[tid] = wacc;
		__syncthreads();
		if (a.wsum && tid == 0) {
			double s = 0.;
			for (int r = 0; r < CH; ++r)
				s += wsh[r];
			a.wsum[blockIdx.x] = a.accumulate ? a.wsum[blockIdx.x] + s : s;
		}
	}
}

template <bool WT, int NI, int NJ>
__global__ __launch_bounds__(kThreads) void rank_update_kernel(Args a)
{
	typedef Pass<NI, NJ> P;
	extern __shared__ double lds[];
	double* wsh = lds;  // after the hand-over
	// wave-uniform branch: waves g and g + 4 run group g
	switch ((threadIdx.x >> 6) & 3) {
	case 0: body<P, WT, 0>(a, lds, wsh); break;
	case 1: body<P, WT, 1>(a, lds, wsh); break;
	case 2: body<P, WT, 2>(a, lds, wsh); break;
	default: body<P, WT, 3>(a, lds, wsh); break;
	}
}

// the passes' kernels: windows of nI and nJ blocks (nJ = 0: the triangle); nJ is nI or one less
struct Kernel {
	void (*k)(Args) = nullptr;
	size_t lds = 0;
};
template <bool WT, int NI, int NJ>
Kernel make()
{
	return Kernel{rank_update_kernel<WT, NI, NJ>, Pass<NI, NJ>::lds};
}
template <bool WT>
Kernel pick(uint32_t nI, uint32_t nJ)
{
	switch (nI * 16 + nJ) {
	case 0x10: return make<WT, 1, 0>();
	case 0x20: return make<WT, 2, 0>();
	case 0x30: return make<WT, 3, 0>();
	case 0x40: return make<WT, 4, 0>();
	case 0x50: return make<WT, 5, 0>();
	case 0x60: return make<WT, 6, 0>();
	case 0x70: return make<WT, 7, 0>();
	case 0x80: return make<WT, 8, 0>();
	case 0x90: return make<WT, 9, 0>();
	case 0xA0: return make<WT, 10, 0>();
	case 0xB0: return make<WT, 11, 0>();
	case 0xC0: return make<WT, 12, 0>();
	case 0x65: return make<WT, 6, 5>();
	case 0x66: return make<WT, 6, 6>();
	case 0x76: return make<WT, 7, 6>();
	case 0x77: return make<WT, 7, 7>();
	case 0x87: return make<WT, 8, 7>();
	case 0x88: return make<WT, 8, 8>();
	default: return Kernel();
	}
}

// window u of nWin over nT blocks: the first nT % nWin are one block longer
inline void window(uint32_t nT, uint32_t nWin, uint32_t u, uint32_t& first, uint32_t& n)
{
	const uint32_t base = nT / nWin, more = nT % nWin;
	first = u * base + std::min(u, more);
	n = base + (u < more ? 1 : 0);
}

// All passes of one update on stream s; winI0, winJ0, nT and nTiles are set here.
template <bool WT>
hipError_t launch(Args a, int nWg, hipStream_t s)
{
	a.nT = (a.D + 15) / 16;
	a.nTiles = a.nT * (a.nT + 1) / 2;
	const uint32_t nWin = a.nT <= (uint32_t)kOneWin ? 1 : (a.nT + kMaxWin - 1) / kMaxWin;
	a.odd = reinterpret_cast<uintptr_t>(a.x) % 16 != 0;
	double* const wsum = a.wsum;
	for (uint32_t u = 0; u < nWin; ++u)
		for (uint32_t v = u; v < nWin; ++v) {
			uint32_t nI, nJ;
			window(a.nT, nWin, u, a.winI0, nI);
			window(a.nT, nWin, v, a.winJ0, nJ);
			const Kernel p = pick<WT>(nI, v > u ? nJ : 0);
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

}  // namespace ru
}  // namespace rpwa_amd
