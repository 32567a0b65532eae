/*
 * tap_product.hpp — one wavefront's product over the nine taps of a 3 x 3 gather and a few channels, operands straight from memory
 * into the registers of the fp32 matrix instruction (the recurrent steps of lstm_steps.hip, the convolutions of few_channels.hip).
 */
#ifndef CATTLE_HIP_TAP_PRODUCT_HPP_
#define CATTLE_HIP_TAP_PRODUCT_HPP_

#include "buffer_loads.hpp"
#include "gemm_tiles.hpp"

#include <algorithm>
#include <cstdlib>

namespace cattle_hip {
namespace tap_product {

using namespace buffer_loads;

typedef Mfma<float>::acc_t acc_t;
constexpr int TAPS = 9;
constexpr int TL = Mfma<float>::TL;

/* n / d for n < 2^31: the host's multiplier in place of a division's two dozen instructions (Granlund and Montgomery, 1994) */
struct Divisor { unsigned mul, shift; };
inline Divisor divisor(unsigned d) {
	unsigned shift = 0;
	while ((1ull << shift) < d)
		++shift;
	return { (unsigned) (((((1ull << shift) - d) << 32) / d) + 1), shift };
}
__device__ __forceinline__ unsigned quotient(unsigned n, Divisor d) {
	return (__umulhi(n, d.mul) + n) >> d.shift;
}

/* What the host works out for a launch. `before` bytes in front of the source are the lowest offset that a tap of a position
 * in the padding would have: the buffer starts there, so that a lane's offset and a tap's are sums of non-negative numbers. */
struct StepGeom {
	Divisor by_N, by_OA;
	unsigned before, src_bytes, wt_bytes;
};

/* The byte offsets of a load, from the start of its buffer: a lane's part (sample n, position a, b; channel slot lk) and the
 * wavefront's, which is the sum of one for its first channel, one for the tap t and one for every pair of channels after the first.
 * A load is in range by what the code says, not by how the hardware compares: the sum of the two parts lies inside the buffer for
 * every lane that takes a value, any other lane is given OUTSIDE, which is beyond every buffer, and the wavefront's part alone never
 * exceeds the buffer's length, so that the difference that OUTSIDE may be compared with is not negative (addressable() asks for that). */
__host__ __device__ __forceinline__ int plane_of(const GatherGeom& g) {
	return g.NS * g.LH * g.LW;
}
__host__ __device__ __forceinline__ unsigned src_lane(const GatherGeom& g, int plane, unsigned n, unsigned a, unsigned b, int lk) {
	return 4u * (n + (unsigned) g.NS * (a + (unsigned) g.LH * b) + (unsigned) (plane * lk));
}
__host__ __device__ __forceinline__ unsigned src_first(const GatherGeom& g, int plane, unsigned before, int channel) {
	return before + 4u * (unsigned) (channel * plane + g.NS * (g.PA + g.LH * g.PB));
}
__host__ __device__ __forceinline__ unsigned src_tap(const GatherGeom& g, int t) {
	return 4u * (unsigned) (g.NS * ((t % 3) * g.RA + g.LH * (t / 3) * g.RB));
}
__host__ __device__ __forceinline__ unsigned wt_lane(const GatherGeom& g, int f, int lk) {
	return 4u * (unsigned) (TAPS * lk * g.ldw + f);
}
__host__ __device__ __forceinline__ unsigned wt_first(const GatherGeom& g, int channel) {
	return 4u * (unsigned) (channel * TAPS * g.ldw);
}
__host__ __device__ __forceinline__ unsigned wt_tap(const GatherGeom& g, int t) {
	return 4u * (unsigned) (t * g.ldw);
}
/* whether tap row r of output row a, tap column s of output column b, lies inside the image */
__host__ __device__ __forceinline__ bool row_inside(const GatherGeom& g, int a, int r) {
	return (unsigned) (a + g.PA + r * g.RA) < (unsigned) g.LH;
}
__host__ __device__ __forceinline__ bool column_inside(const GatherGeom& g, int b, int s) {
	return (unsigned) (b + g.PB + s * g.RB) < (unsigned) g.LW;
}

/* The row m of this lane as sample and position. */
struct Row { unsigned n, pos, a, b; };
__device__ __forceinline__ Row row_of(unsigned m, const GatherGeom& g, const StepGeom& G) {
	Row r;
	r.pos = quotient(m, G.by_N);
	r.n = m - r.pos * (unsigned) g.N;
	r.b = quotient(r.pos, G.by_OA);
	r.a = r.pos - r.b * (unsigned) g.OA;
	return r;
}

/* One wavefront's share of the product for a tile of 32 rows and 32 columns: 2 SPC channels from `channel` on, all nine taps.
 * The lane that holds row lane % 32 and column f_lane loads for channel slot lane / 32, straight into the operands' registers. A
 * load's address is one register (OUTSIDE or a lane's own offset, by whether the tap falls into the padding) and one scalar. ODD: the
 * second channel of the last pair does not exist. */
template<int SPC, bool ODD = false>
__device__ __forceinline__ acc_t share_of_product(const float* __restrict__ src, const float* __restrict__ wt, const GatherGeom& g,
		const StepGeom& G, const Row& row, bool valid, int lk, int f_lane, int channel) {
	const __amdgpu_buffer_rsrc_t src_buf = buffer_of(reinterpret_cast<const char*>(src) - G.before, G.src_bytes);
	const __amdgpu_buffer_rsrc_t wt_buf = buffer_of(wt, G.wt_bytes);
	const int plane = plane_of(g);
	const unsigned a_lane = src_lane(g, plane, row.n, row.a, row.b, lk);
	const unsigned b_lane = wt_lane(g, f_lane, lk);
	const bool missing = ODD && lk == 1;
	bool in_a[3], in_b[3];
	#pragma unroll
	for (int r = 0; r < 3; ++r) {
		in_a[r] = valid && row_inside(g, (int) row.a, r);
		in_b[r] = column_inside(g, (int) row.b, r);
	}
	const unsigned a_pair = 8u * (unsigned) plane, b_pair = 8u * (unsigned) (TAPS * g.ldw);
	const unsigned a_wave = src_first(g, plane, G.before, channel);
	const unsigned b_wave = wt_first(g, channel);
	acc_t acc;
	#pragma unroll
	for (int r = 0; r < 16; ++r)
		acc[r] = 0.f;
	/* All loads of up to 36 steps are issued, then the products run as the values arrive: one round trip to memory per
	 * wavefront, where batches that followed each other were two or three (a wavefront has 128 registers; nothing else of
	 * the block runs on the CU that could hide them). */
	constexpr int BATCH = SPC <= 4 ? TAPS : 5;
	#pragma unroll
	for (int t0 = 0; t0 < TAPS; t0 += BATCH) {
		float x[BATCH * SPC], w[BATCH * SPC];
		#pragma unroll
		for (int j = 0; j < BATCH; ++j) {
			const int t = t0 + j;
			if (t < TAPS) {
				const unsigned lane_off = in_a[t % 3] && in_b[t / 3] ? a_lane : OUTSIDE;
				const unsigned a_tap = a_wave + src_tap(g, t);
				#pragma unroll
				for (int i = 0; i < SPC; ++i) {
					const bool last = ODD && i == SPC - 1;
					x[j * SPC + i] = load_1(src_buf, last && missing ? OUTSIDE : lane_off, a_tap + (unsigned) i * a_pair);
					w[j * SPC + i] = load_1(wt_buf, last && missing ? OUTSIDE : b_lane, b_wave + wt_tap(g, t) + (unsigned) i * b_pair);
				}
				/* in the order of the products: left alone, the compiler issues the last channel's loads behind all others (both passes of
				 * 65,536 x 27 x 16 20.5 us, 19.7 this way) */
				if constexpr (ODD)
					__builtin_amdgcn_sched_barrier(0);
			}
		}
		__builtin_amdgcn_sched_barrier(0);
		#pragma unroll
		for (int j = 0; j < BATCH; ++j)
			if (t0 + j < TAPS) {
				#pragma unroll
				for (int i = 0; i < SPC; ++i)
					acc = Mfma<float>::mma(w[j * SPC + i], x[j * SPC + i], acc);
			}
		__builtin_amdgcn_sched_barrier(0);
	}
	return acc;
}

/* Offsets of 32 bits, and nothing that share_of_product does not know: strides, divisors, other receptors, images so small that the last
 * tap reaches as far past a channel as the whole of it (a side of one, or of two with dilation) where no channel of the pair follows */
inline bool addressable(const GatherGeom& g) {
	const double bytes = 4.0 * g.NS * g.LH * g.LW * g.LC, wt_bytes = 4.0 * (g.R * g.S * (double) g.LC) * g.ldw;
	const double before = 4.0 * g.NS * (2.0 * std::abs(g.RA) + std::abs(g.PA) + g.LH * (2.0 * std::abs(g.RB) + std::abs(g.PB)));
	const double highest = g.PA + std::max(0, 2 * g.RA) + (double) g.LH * (g.PB + std::max(0, 2 * g.RB));
	return g.R == 3 && g.S == 3 && g.SA == 1 && g.SB == 1 && g.DA == 1 && g.DB == 1 && bytes + 2 * before < 2147483648.0 && wt_bytes < 2147483648.0 &&
			highest <= (double) g.LH * g.LW * (g.LC - (g.LC - 1) / 2 * 2);
}
inline StepGeom step_geom(const GatherGeom& g) {
	const int lowest = g.NS * ((g.PA + std::min(0, 2 * g.RA)) + g.LH * (g.PB + std::min(0, 2 * g.RB)));
	StepGeom G;
	G.by_N = divisor((unsigned) g.N);
	G.by_OA = divisor((unsigned) g.OA);
	G.before = lowest < 0 ? 4u * (unsigned) -lowest : 0u;
	G.src_bytes = G.before + 4u * (unsigned) (g.NS * g.LH * g.LW) * (unsigned) g.LC;
	G.wt_bytes = 4u * (unsigned) (TAPS * g.LC) * (unsigned) g.ldw;
	return G;
}
inline int tiles_of(int n) {
	return (n + TL - 1) / TL;
}

} /* namespace tap_product */
} /* namespace cattle_hip */

#endif /* CATTLE_HIP_TAP_PRODUCT_HPP_ */
