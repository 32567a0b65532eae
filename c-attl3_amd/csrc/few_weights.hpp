/*
 * few_weights.hpp — the fp32 weight gradient of layers with few weights over many positions (the first layer of an image network,
 * the layers of an autoencoder): the body of its kernel, which is also one of a launch that takes it along, and its own launch
 * (few_weights.hip).
 */
#ifndef CATTLE_HIP_FEW_WEIGHTS_HPP_
#define CATTLE_HIP_FEW_WEIGHTS_HPP_

#include "buffer_loads.hpp"
#include "gemm_tiles.hpp"

namespace cattle_hip {
namespace few_weights {

using namespace buffer_loads;

constexpr int TL = 32, ITEM = 64, HALF = 32, ROWS = 64 / UNITS;
constexpr int WAVES = 4;        /* of a block, alone and riding: the order of the sums does not depend on which */
static_assert(UNITS == HALF / 4, "rows of 32 samples");

/* ------------------------------------------------------------------------------------------------
 * partials[slice][K x F] = sum over the slice of x^T og. An item is 64 samples of one output position; a slice is a block, its
 * wavefronts take its items in turn, 32 weights (rows) by all filters (columns, up to 32) each, and their sums meet in LDS. All loads
 * of an item are issued at once, eight lanes to the 32 samples of a row (whole lines), and the operands turn in LDS into the
 * matrix instruction's layout, in which a lane holds a row.
 * Bound by latency: wgrad_kernel's blocks are one wavefront that walks its slice in chunks of 32 rows, a round trip to memory each.
 * 43,264 x 16 x 3 13.4 -> 5.6 us, 25,600 x 48 x 3 13.1 -> 5.6, and in the launch of its input gradient 14.7 -> 6.7; 65,536 x 27 x 16
 * with its input gradient 11.0 -> 9.0.
 * ---------------------------------------------------------------------------------------------- */
struct FewWeights {
	const float *x, *og;
	float *partials, *bias_partials;
	GatherGeom g;
	int items, groups, per_slice, slices;
	bool transposed;        /* a slice is F x K, not K x F */
	unsigned x_bytes, og_bytes;
};
/* stage: 8 KB per wavefront of the block: [wavefront][x, og][row][unit], then partial tiles and column sums */
template<int GQ>
__device__ __forceinline__ void few_weights_body(const FewWeights& A, int slice, int k_tile, f32x4* stage) {
	const GatherGeom& g = A.g;
	const float* __restrict__ const x = A.x;
	const float* __restrict__ const og = A.og;
	const int groups = A.groups;
	const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), waves = blockDim.x / 64;
	const int k0 = k_tile * TL;
	const int lc = lane % TL, lk = lane / TL, row = lane / UNITS, unit = lane % UNITS;
	const __amdgpu_buffer_rsrc_t x_buf = buffer_of(x, A.x_bytes), og_buf = buffer_of(og, A.og_bytes);
	/* this lane's rows of the weight matrix: receptor position and channel */
	constexpr int Q = TL / ROWS;
	const int taps = g.R * g.S, plane = g.NS * g.LH * g.LW;
	int da[Q], db[Q], offset[Q];
	#pragma unroll
	for (int q = 0; q < Q; ++q) {
		const int k = k0 + row + ROWS * q, c = k / taps, tap = k - c * taps, s = tap / g.R;
		da[q] = (tap - s * g.R) * g.RA + g.PA;
		db[q] = s * g.RB + g.PB;
		offset[q] = k < g.K ? 4 * (g.NS * (da[q] + g.LH * db[q]) + plane * c) : 0;
		if (k >= g.K)
			da[q] = -0x40000000;            /* never inside */
	}
	typename Mfma<float>::acc_t acc;
	#pragma unroll
	for (int r = 0; r < 16; ++r)
		acc[r] = 0.f;
	float bias[GQ];
	#pragma unroll
	for (int q = 0; q < GQ; ++q)
		bias[q] = 0.f;
	f32x4* const xs = stage + wave * 2 * TL * UNITS;
	f32x4* const zs = xs + TL * UNITS;
	/* the columns past the filters' eights are zero throughout */
	#pragma unroll
	for (int q = GQ; q < Q; ++q)
		zs[unit_of(row + ROWS * q, unit)] = (f32x4) { 0.f, 0.f, 0.f, 0.f };

	const int end = min(A.items, (slice + 1) * A.per_slice);
	for (int item = slice * A.per_slice + wave; item < end; item += waves) {
		const int pos = item / groups, n0 = (item - pos * groups) * ITEM;
		const int b = pos / g.OA, a = pos - b * g.OA;
		const int ya0 = a * g.SA, yb0 = b * g.SB;
		const int x_pos = 4 * (g.NS * (ya0 + g.LH * yb0) + n0), og_pos = 4 * (g.N * pos + n0);
		f32x4 xv[2][Q], gv[2][GQ];
		#pragma unroll
		for (int h = 0; h < 2; ++h) {
			const int n = 4 * unit + HALF * h;
			const bool in = n0 + n < g.N;
			#pragma unroll
			for (int q = 0; q < GQ; ++q)
				gv[h][q] = load_4(og_buf, in && row + ROWS * q < g.F ? 4u * (unsigned) (n + (row + ROWS * q) * g.M) : OUTSIDE, (unsigned) og_pos);
			#pragma unroll
			for (int q = 0; q < Q; ++q) {
				const bool ok = in && (unsigned) (ya0 + da[q]) < (unsigned) g.LH && (unsigned) (yb0 + db[q]) < (unsigned) g.LW;
				xv[h][q] = load_4(x_buf, ok ? (unsigned) (x_pos + offset[q] + 4 * n) : OUTSIDE, 0u);
			}
		}
		__builtin_amdgcn_sched_barrier(0);
		#pragma unroll
		for (int h = 0; h < 2; ++h) {
			#pragma unroll
			for (int q = 0; q < GQ; ++q) {
				zs[unit_of(row + ROWS * q, unit)] = gv[h][q];
				#pragma unroll
				for (int i = 0; i < 4; ++i)
					bias[q] += gv[h][q][i];
			}
			#pragma unroll
			for (int q = 0; q < Q; ++q)
				xs[unit_of(row + ROWS * q, unit)] = xv[h][q];
			/* (the wavefront's own region: its LDS instructions run in order) */
			__builtin_amdgcn_wave_barrier();
			#pragma unroll
			for (int q = 0; q < UNITS / 2; ++q) {
				const f32x4 z4 = zs[unit_of(lc, 2 * q + lk)], x4 = xs[unit_of(lc, 2 * q + lk)];
				#pragma unroll
				for (int i = 0; i < 4; ++i)
					acc = Mfma<float>::mma(z4[i], x4[i], acc);
			}
			__builtin_amdgcn_wave_barrier();
		}
	}
	float* const part = reinterpret_cast<float*>(xs);
	#pragma unroll
	for (int r = 0; r < 16; ++r)
		part[acc_row<float>(r, lk) * TL + lc] = acc[r];
	const bool sums_bias = k_tile == 0 && A.bias_partials != nullptr;
	if (sums_bias) {
		#pragma unroll
		for (int q = 0; q < GQ; ++q) {
			#pragma unroll
			for (int off = 1; off < UNITS; off *= 2)
				bias[q] += __shfl_xor(bias[q], off, 64);
			if (unit == 0)
				part[TL * TL + row + ROWS * q] = bias[q];
		}
	}
	__syncthreads();
	constexpr int STRIDE = 2 * TL * TL;
	const float* const red = reinterpret_cast<const float*>(stage);
	float* const dst = A.partials + (size_t) slice * ((size_t) g.K * g.F);
	for (int o = tid; o < TL * 8 * GQ; o += blockDim.x) {
		float v = red[o];
		for (int w = 1; w < waves; ++w)
			v += red[w * STRIDE + o];
		const int k = k0 + o % TL, f = o / TL;
		if (k < g.K && f < g.F)
			dst[A.transposed ? (size_t) f + (size_t) g.F * k : (size_t) k + (size_t) g.K * f] = v;
	}
	if (sums_bias && tid < g.F) {
		float v = red[TL * TL + tid];
		for (int w = 1; w < waves; ++w)
			v += red[w * STRIDE + TL * TL + tid];
		A.bias_partials[(size_t) slice * g.F + tid] = v;
	}
}

} /* namespace few_weights */

/* Whether the weight gradient of this forward gather is one of few_weights_gradient's (operands on 16-byte boundaries and g.N a
 * multiple of four: `vec`). */
bool few_weights_possible(const GatherGeom& g, bool vec);
/* The slices it writes, at most `most`. */
int few_weights_slices(const GatherGeom& g, int most);
/* partials[slice][K x F], bias_partials[slice][F] (or null): the sums of x^T og and of og over the slice's rows */
few_weights::FewWeights few_weights_problem(const float* x, const float* og, float* partials, float* bias_partials, const GatherGeom& g, int slices,
		bool transposed = false);
void few_weights_gradient(const few_weights::FewWeights& problem);

} /* namespace cattle_hip */

#endif /* CATTLE_HIP_FEW_WEIGHTS_HPP_ */
