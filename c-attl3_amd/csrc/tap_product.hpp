/*
 * tap_product.hpp — one wavefront's product over the nine taps of a 3 x 3 gather and a few channels, operands straight from memory
 * into the registers of the fp32 matrix instruction (the recurrent steps of lstm_steps.hip, the convolutions of few_channels.hip).
 */
#ifndef CATTLE_HIP_TAP_PRODUCT_HPP_
#define CATTLE_HIP_TAP_PRODUCT_HPP_

#include "gemm_tiles.hpp"

#include <cstdlib>

namespace cattle_hip {
namespace tap_product {

typedef Mfma<float>::acc_t acc_t;
constexpr int TAPS = 9;
constexpr int TL = Mfma<float>::TL;
constexpr unsigned OUTSIDE = 0x80000000u;       /* a byte offset beyond any buffer: such a load returns zero */

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

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, unsigned bytes) {
	return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int) bytes, 0x00020000);
}
__device__ __forceinline__ float load_f32(__amdgpu_buffer_rsrc_t b, unsigned lane_off, unsigned wave_off) {
	return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, (int) lane_off, (int) wave_off, 0));
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
 * load's address is one register (zero or a lane's own offset, by whether the tap falls into the padding) and one scalar. */
template<int SPC>
__device__ __forceinline__ acc_t share_of_product(const float* __restrict__ src, const float* __restrict__ wt, const GatherGeom& g,
		const StepGeom& G, const Row& row, bool valid, int lk, int f_lane, int channel) {
	const __amdgpu_buffer_rsrc_t src_buf = buffer_of(reinterpret_cast<const char*>(src) - G.before, G.src_bytes);
	const __amdgpu_buffer_rsrc_t wt_buf = buffer_of(wt, G.wt_bytes);
	const int plane = g.NS * g.LH * g.LW;
	const unsigned a_lane = 4u * (row.n + (unsigned) g.NS * (row.a + (unsigned) g.LH * row.b) + (unsigned) (plane * lk));
	const unsigned b_lane = 4u * (unsigned) (TAPS * lk * g.ldw + f_lane);
	bool in_a[3], in_b[3];
	#pragma unroll
	for (int r = 0; r < 3; ++r) {
		in_a[r] = valid && (unsigned) ((int) row.a + g.PA + r * g.RA) < (unsigned) g.LH;
		in_b[r] = (unsigned) ((int) row.b + g.PB + r * g.RB) < (unsigned) g.LW;
	}
	const unsigned a_channel = 8u * (unsigned) plane, b_channel = 8u * (unsigned) (TAPS * g.ldw);
	const unsigned a_wave = G.before + 4u * (unsigned) (channel * plane + g.NS * (g.PA + g.LH * g.PB));
	const unsigned b_wave = 4u * (unsigned) (channel * TAPS * g.ldw);
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
				const unsigned a_tap = a_wave + 4u * (unsigned) (g.NS * ((t % 3) * g.RA + g.LH * (t / 3) * g.RB));
				#pragma unroll
				for (int i = 0; i < SPC; ++i) {
					x[j * SPC + i] = load_f32(src_buf, lane_off, a_tap + (unsigned) i * a_channel);
					w[j * SPC + i] = load_f32(wt_buf, b_lane, b_wave + 4u * (unsigned) (t * g.ldw) + (unsigned) i * b_channel);
				}
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

/* Offsets of 32 bits, and nothing that share_of_product does not know: strides, divisors, other receptors */
inline bool addressable(const GatherGeom& g) {
	const double bytes = 4.0 * g.NS * g.LH * g.LW * g.LC, wt_bytes = 4.0 * (g.R * g.S * (double) g.LC) * g.ldw;
	const double before = 4.0 * g.NS * (2.0 * std::abs(g.RA) + std::abs(g.PA) + g.LH * (2.0 * std::abs(g.RB) + std::abs(g.PB)));
	return g.R == 3 && g.S == 3 && g.SA == 1 && g.SB == 1 && g.DA == 1 && g.DB == 1 && bytes + 2 * before < 2147483648.0 && wt_bytes < 2147483648.0;
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
