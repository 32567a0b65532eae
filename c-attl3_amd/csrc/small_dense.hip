/*
 * small_dense.hip — fp32 matrix products of dense layers with few output tiles: one launch, one round trip to memory. Matrices are
 * column-major as everywhere: x is M x K with the samples (rows) contiguous.
 */
#include "small_dense.hpp"
#include "act_math.hpp"
#include "buffer_loads.hpp"

namespace cattle_hip {
namespace {

using namespace buffer_loads;

/* ------------------------------------------------------------------------------------------------
 * out[M x F] = x[M x K] wt[K x F] (+ bias, activation). A block owns 16 MB rows and 16 columns, and its wavefronts a contiguous
 * share of the reduction each, whose operands go straight from memory into the registers of the 16 x 16 x 4 instruction, up to
 * sixteen steps (64 reduction indices) in flight; the partial tiles meet in LDS and are added in a fixed order.
 * Bound by latency: a launch, a round trip to memory, the sum. Against wave_split_gemm_kernel, whose 32 x 32 tiles gave 128 CUs
 * 2.6 us of matrix instructions each and left the others idle, and which fetched the bias after the reduction: 256 x 784 -> 512
 * 9.9 -> 5.2 us, 256 x 512 -> 256 7.4 -> 4.6, 256 x 256 -> 10 6.4 -> 3.8, one sample of 784 -> 512 8.0 -> 5.2, and with its
 * activation at any batch size (the 16-byte accesses of the tiled launches need a multiple of four).
 * ---------------------------------------------------------------------------------------------- */
constexpr int PL = 16, PK = 4, MAX_STEPS = 16;
constexpr int chains(int mb) { return mb == 1 ? 8 : 4; }
struct ProductArgs {
	int M, K, F, ldw, mtiles, tiles, per;          /* per: steps of the reduction per wavefront */
	unsigned x_bytes, wt_bytes;
	int kind;                                       /* activation, or -1 */
	float p;
	float* pre;
};

__device__ __forceinline__ void finish_product(const ProductArgs& A, float* __restrict__ out, int m, int f, float v) {
	const size_t at = (size_t) m + (size_t) A.M * f;
	if (A.kind >= 0) {
		if (A.pre)
			A.pre[at] = v;
		act_dispatch(A.kind, [&](auto kc) {
			v = act_f_coded<float, decltype(kc)::value>(v, A.p);
		});
	}
	__builtin_nontemporal_store(v, out + at);
}

/* PAIRS: rows 2 l and 2 l + 1 of a tile belong to lane l, one load of eight bytes; else rows l and l + 16. x_last: the offsets of the last
 * of the steps, which are those of the others unless TAIL. */
template<int MB, bool PAIRS, bool TAIL, int STEPS>
__device__ __forceinline__ void product_steps(f32x4 (&acc)[chains(MB)][MB], __amdgpu_buffer_rsrc_t x_buf, __amdgpu_buffer_rsrc_t wt_buf,
		const unsigned (&x_lane)[MB], const unsigned (&x_last)[MB], unsigned w_lane, unsigned x_wave, unsigned w_wave, unsigned x_step,
		unsigned w_step) {
	float x[STEPS][MB], w[STEPS];
	#pragma unroll
	for (int s = 0; s < STEPS; ++s) {
		w[s] = load_1(wt_buf, w_lane, w_wave + (unsigned) s * w_step);
		if constexpr (PAIRS) {
			const f32x2 v = load_2(x_buf, TAIL && s == STEPS - 1 ? x_last[0] : x_lane[0], x_wave + (unsigned) s * x_step);
			x[s][0] = v[0];
			x[s][MB - 1] = v[1];
		} else {
			#pragma unroll
			for (int j = 0; j < MB; ++j)
				x[s][j] = load_1(x_buf, TAIL && s == STEPS - 1 ? x_last[j] : x_lane[j], x_wave + (unsigned) s * x_step);
		}
	}
	__builtin_amdgcn_sched_barrier(0);
	#pragma unroll
	for (int s = 0; s < STEPS; ++s)
		#pragma unroll
		for (int j = 0; j < MB; ++j)
			acc[s % chains(MB)][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s], x[s][j], acc[s % chains(MB)][j], 0, 0, 0);
	__builtin_amdgcn_sched_barrier(0);
}

/* TAIL: the reduction ends inside a step. (With that select in every launch, and one for rows past M in the place of the last row read
 * again, here and below, a training pass of 784-512-256-10, eight batches of 256, takes 420 us instead of 417.) */
template<int MB, bool PAIRS, bool TAIL>
__global__ __launch_bounds__(1024)
void small_product_kernel(const float* __restrict__ src, const float* __restrict__ wt, const float* __restrict__ bias, float* __restrict__ out,
		const ProductArgs A) {
	static_assert(!PAIRS || MB == 2, "a pair of rows is two row blocks");
	constexpr int BM = PL * MB;
	__shared__ float red[16 * PL * BM];             /* [wavefront][column][row] */
	/* column tiles outermost: an XCD then reads few columns of the weights and all rows, which are fewer */
	const int tile = xcd_tile(blockIdx.x, A.tiles);
	if (tile >= A.tiles)
		return;
	const int mt = tile % A.mtiles, m0 = mt * BM, f0 = tile / A.mtiles * PL;
	const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), waves = blockDim.x / 64;
	const int lc = lane % PL, lk = lane / PL;
	/* the bias of this thread's output is fetched now: after the reduction it would be a round trip to memory of its own */
	const int of = f0 + tid / BM;
	const float bv = bias != nullptr && of < A.F ? bias[of] : 0.f;

	const __amdgpu_buffer_rsrc_t x_buf = buffer_of(src, A.x_bytes), wt_buf = buffer_of(wt, A.wt_bytes);
	const int total = (A.K + PK - 1) / PK;
	int s = wave * A.per;
	const int end = min(total, s + A.per);
	const unsigned x_step = 4u * PK * (unsigned) A.M, w_step = 4u * PK * (unsigned) A.ldw;
	/* (rows past M are the last one again, and nobody stores them; reduction indices past K are zeros; the weights have rows for all
	 * steps and columns for all tiles) */
	unsigned x_lane[MB], x_last[MB];
	#pragma unroll
	for (int j = 0; j < MB; ++j)
		x_lane[j] = 4u * (unsigned) (min(m0 + (PAIRS ? 2 * lc : lc + PL * j), A.M - (PAIRS ? 2 : 1)) + lk * A.M);
	const unsigned w_lane = 4u * (unsigned) (f0 + lc + lk * A.ldw);
	/* Every fourth (eighth) step goes to an accumulator of its own, so that a sum is rounded as often as one of a fraction of the
	 * length. Error of the output against 64 bits in the 2-norm, with one, and with these: 256 x 784 -> 512 1.5e-7, 1.0e-7; 128 x 3000 ->
	 * 128 2.6e-7, 1.2e-7 (1.2e-7 on the bf16 instructions). */
	constexpr int CHAINS = chains(MB);
	f32x4 sums[CHAINS][MB];
	#pragma unroll
	for (int c = 0; c < CHAINS; ++c)
		#pragma unroll
		for (int j = 0; j < MB; ++j)
			sums[c][j] = (f32x4) { 0.f, 0.f, 0.f, 0.f };
	while (s < end) {
		const int steps = min(end - s, MAX_STEPS);
		const unsigned x_wave = (unsigned) s * x_step, w_wave = (unsigned) s * w_step;
		#pragma unroll
		for (int j = 0; j < MB; ++j)
			x_last[j] = TAIL && s + steps == total && PK * (total - 1) + lk >= A.K ? OUTSIDE : x_lane[j];
		switch (steps) {
#define CATTLE_HIP_STEPS(n) case n: product_steps<MB, PAIRS, TAIL, n>(sums, x_buf, wt_buf, x_lane, x_last, w_lane, x_wave, w_wave, x_step, w_step); break;
		CATTLE_HIP_STEPS(1) CATTLE_HIP_STEPS(2) CATTLE_HIP_STEPS(3) CATTLE_HIP_STEPS(4) CATTLE_HIP_STEPS(5) CATTLE_HIP_STEPS(6)
		CATTLE_HIP_STEPS(7) CATTLE_HIP_STEPS(8) CATTLE_HIP_STEPS(9) CATTLE_HIP_STEPS(10) CATTLE_HIP_STEPS(11) CATTLE_HIP_STEPS(12)
		CATTLE_HIP_STEPS(13) CATTLE_HIP_STEPS(14) CATTLE_HIP_STEPS(15)
		default: product_steps<MB, PAIRS, TAIL, MAX_STEPS>(sums, x_buf, wt_buf, x_lane, x_last, w_lane, x_wave, w_wave, x_step, w_step);
#undef CATTLE_HIP_STEPS
		}
		s += steps;
	}
	f32x4 acc[MB];
	#pragma unroll
	for (int j = 0; j < MB; ++j)
		acc[j] = (sums[0][j] + sums[1][j]) + (sums[2][j] + sums[3][j]);
	if constexpr (CHAINS == 8)
		acc[0] += (sums[4][0] + sums[5][0]) + (sums[6][0] + sums[7][0]);
	#pragma unroll
	for (int r = 0; r < 4; ++r) {
		float* dst = red + (wave * PL + 4 * lk + r) * BM;
		if constexpr (PAIRS) {
			*reinterpret_cast<f32x2*>(dst + 2 * lc) = (f32x2) { acc[0][r], acc[MB - 1][r] };
		} else {
			#pragma unroll
			for (int j = 0; j < MB; ++j)
				dst[lc + PL * j] = acc[j][r];
		}
	}
	__syncthreads();
	for (int o = tid; o < PL * BM; o += blockDim.x) {
		/* (in four sums again, for the same reason) */
		float part[4] = { 0.f, 0.f, 0.f, 0.f };
		if (waves == 16) {
			#pragma unroll
			for (int w = 0; w < 16; ++w)
				part[w % 4] += red[w * PL * BM + o];
		} else
			for (int w = 0; w < waves; ++w) {
				part[3] += red[w * PL * BM + o];
				const float first = part[0];
				part[0] = part[1];
				part[1] = part[2];
				part[2] = part[3];
				part[3] = first;
			}
		float v = (part[0] + part[1]) + (part[2] + part[3]);
		const int m = m0 + o % BM, f = f0 + o / BM;
		if (m >= A.M || f >= A.F)
			continue;
		v += o == tid ? bv : (bias != nullptr ? bias[f] : 0.f);
		finish_product(A, out, m, f, v);
	}
}

/* The same product with its sums in the order of wave_split_gemm_kernel (GatherProblem::keeps_sums), bit for bit: 32 x 32 tiles of the
 * 32 x 32 x 2 instruction, one accumulator a wavefront, the same shares, added in ascending order and the bias last. What differs
 * is the wait: one address register and one scalar per load, up to 32 steps in flight whatever their number, and the bias of an
 * output fetched before the reduction. 128 of the 256 CUs have a tile of 256 x 784 -> 512, with 2.6 us of matrix
 * instructions: 9.9 -> 8.6 us; 256 x 512 -> 256 7.4 -> 6.5. */
constexpr int OL = 32, OK = 2, MAX_ORDERED = 32;
template<int STEPS>
__device__ __forceinline__ void ordered_steps(Mfma<float>::acc_t& acc, __amdgpu_buffer_rsrc_t x_buf, __amdgpu_buffer_rsrc_t wt_buf,
		unsigned x_lane, unsigned w_lane, unsigned x_wave, unsigned w_wave, unsigned x_step, unsigned w_step) {
	float x[STEPS], w[STEPS];
	#pragma unroll
	for (int s = 0; s < STEPS; ++s) {
		w[s] = load_1(wt_buf, w_lane, w_wave + (unsigned) s * w_step);
		x[s] = load_1(x_buf, x_lane, x_wave + (unsigned) s * x_step);
	}
	__builtin_amdgcn_sched_barrier(0);
	#pragma unroll
	for (int s = 0; s < STEPS; ++s)
		acc = Mfma<float>::mma(w[s], x[s], acc);
	__builtin_amdgcn_sched_barrier(0);
}
__global__ __launch_bounds__(1024)
void small_product_ordered_kernel(const float* __restrict__ src, const float* __restrict__ wt, const float* __restrict__ bias,
		float* __restrict__ out, const ProductArgs A) {
	__shared__ float red[16 * OL * OL];             /* [wavefront][column][row] */
	const int tile = xcd_tile(blockIdx.x, A.tiles);
	if (tile >= A.tiles)
		return;
	const int m0 = tile % A.mtiles * OL, f0 = tile / A.mtiles * OL;
	const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), waves = blockDim.x / 64;
	const int lc = lane % OL, lk = lane / OL;
	const int of = f0 + tid / OL;
	const float bv = bias != nullptr && of < A.F ? bias[of] : 0.f;
	const __amdgpu_buffer_rsrc_t x_buf = buffer_of(src, A.x_bytes), wt_buf = buffer_of(wt, A.wt_bytes);
	int s = wave * A.per;
	const int end = min(A.K / OK, s + A.per);
	const unsigned x_step = 4u * OK * (unsigned) A.M, w_step = 4u * OK * (unsigned) A.ldw;
	/* (rows past M are the last one again, and nobody stores them) */
	const unsigned x_lane = 4u * (unsigned) (min(m0 + lc, A.M - 1) + lk * A.M), w_lane = 4u * (unsigned) (f0 + lc + lk * A.ldw);
	Mfma<float>::acc_t acc;
	#pragma unroll
	for (int r = 0; r < 16; ++r)
		acc[r] = 0.f;
	while (s < end) {
		const int steps = min(end - s, MAX_ORDERED);
		const unsigned x_wave = (unsigned) s * x_step, w_wave = (unsigned) s * w_step;
		switch (steps) {
#define CATTLE_HIP_STEPS(n) case n: ordered_steps<n>(acc, x_buf, wt_buf, x_lane, w_lane, x_wave, w_wave, x_step, w_step); break;
#define CATTLE_HIP_EIGHT_STEPS(n) CATTLE_HIP_STEPS(n) CATTLE_HIP_STEPS(n + 1) CATTLE_HIP_STEPS(n + 2) CATTLE_HIP_STEPS(n + 3) \
		CATTLE_HIP_STEPS(n + 4) CATTLE_HIP_STEPS(n + 5) CATTLE_HIP_STEPS(n + 6) CATTLE_HIP_STEPS(n + 7)
		CATTLE_HIP_EIGHT_STEPS(1) CATTLE_HIP_EIGHT_STEPS(9) CATTLE_HIP_EIGHT_STEPS(17) CATTLE_HIP_EIGHT_STEPS(25)
#undef CATTLE_HIP_EIGHT_STEPS
#undef CATTLE_HIP_STEPS
		}
		s += steps;
	}
	#pragma unroll
	for (int r = 0; r < 16; ++r)
		red[(wave * OL + acc_row<float>(r, lk)) * OL + lc] = acc[r];
	__syncthreads();
	for (int o = tid; o < OL * OL; o += blockDim.x) {
		float v = red[o];
		for (int w = 1; w < waves; ++w)
			v += red[w * OL * OL + o];
		const int m = m0 + o % OL, f = f0 + o / OL;
		if (m >= A.M || f >= A.F)
			continue;
		v += o == tid ? bv : (bias != nullptr ? bias[f] : 0.f);
		finish_product(A, out, m, f, v);
	}
}

/* ------------------------------------------------------------------------------------------------
 * wgrad[K x F] += x^T z, bgrad[F] += column sums of z, z = og or slope(y) * og. A block owns a 32 x 32 tile and each of its
 * wavefronts 32 or 64 samples: all its loads are issued at once, the operands change places through LDS (a lane of the instruction holds
 * a column, a line of memory 32 samples of one: 256 x 784 x 512 with the lanes reading their own columns 11.2 us, 7.7 this way),
 * and the wavefronts' sums meet in LDS and are added to the gradient in ascending order. No slices of M in memory: wgrad_kernel took
 * 9.3 us there and left four slices for the optimizer to add (11.6 us, 7.8 without them). A batch of up to eight wavefronts'
 * shares; with 32 columns or more, so that no tile is mostly padding (a layer of few outputs has a launch
 * that its input gradient takes along).
 * ---------------------------------------------------------------------------------------------- */
constexpr int GL = 32, HALF_M = 32, GRAD_WAVES = 8;
static_assert(UNITS == HALF_M / 4, "rows of 32 samples");
/* HALVES: 32 samples each that a wavefront takes */
template<bool ACT, int HALVES>
__global__ __launch_bounds__(64 * GRAD_WAVES)
void small_weight_gradient_kernel(const float* __restrict__ x, const float* __restrict__ og, float* __restrict__ wgrad, float* __restrict__ bgrad,
		int M, int K, int F, int ktiles, int tiles, unsigned x_bytes, unsigned og_bytes, const float* __restrict__ act_y, float* __restrict__ act_dz,
		float p0, float p1, bool fresh) {
	constexpr int ROWS = 64 / UNITS, LOADS = GL / ROWS;             /* rows per load of a wavefront, loads per operand and half */
	/* a wavefront's half shares of x and z; then its partial tile in the place of x and its column sums in that of z */
	extern __shared__ f32x4 stage[];                                /* [wavefront][x, z][column][unit] */
	static_assert(4 * GL * UNITS == GL * GL, "the partial tile takes the place of x");
	const int tile = xcd_tile(blockIdx.x, tiles);
	if (tile >= tiles)
		return;
	const int kt = tile % ktiles, k0 = kt * GL, f0 = tile / ktiles * GL;
	const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), waves = blockDim.x / 64;
	const int lc = lane % GL, lk = lane / GL;
	const __amdgpu_buffer_rsrc_t x_buf = buffer_of(x, x_bytes), og_buf = buffer_of(og, og_bytes), y_buf = buffer_of(ACT ? act_y : og, og_bytes);
	/* loads: eight lanes read 32 samples of a column, whole lines */
	const int row = lane / UNITS, unit = lane % UNITS, m0 = wave * HALVES * HALF_M + 4 * unit;
	const unsigned x_lane = 4u * (unsigned) (M * (k0 + row) + m0), g_lane = 4u * (unsigned) (M * (f0 + row) + m0), rows = 4u * ROWS * (unsigned) M;
	f32x4 xv[HALVES][LOADS], gv[HALVES][LOADS], yv[ACT ? HALVES : 1][LOADS];
	#pragma unroll
	for (int h = 0; h < HALVES; ++h) {
		const bool in = m0 + h * HALF_M < M;
		const unsigned half = 4u * HALF_M * (unsigned) h;
		#pragma unroll
		for (int q = 0; q < LOADS; ++q) {
			const unsigned at = half + rows * (unsigned) q;
			const unsigned xo = in && k0 + row + ROWS * q < K ? x_lane + at : OUTSIDE, go = in && f0 + row + ROWS * q < F ? g_lane + at : OUTSIDE;
			gv[h][q] = load_4(og_buf, go, 0u);
			if constexpr (ACT)
				yv[h][q] = load_4(y_buf, go, 0u);
			xv[h][q] = load_4(x_buf, xo, 0u);
		}
	}
	/* the gradient that the sums are added to, fetched with the operands: up to four values a thread, all of them from 256 threads on */
	float before[4];
	#pragma unroll
	for (int i = 0; i < 4; ++i) {
		const int o = tid + i * (int) blockDim.x, k = k0 + o % GL, f = f0 + o / GL;
		before[i] = !fresh && o < GL * GL && k < K && f < F ? wgrad[(size_t) k + (size_t) K * f] : 0.f;
	}
	__builtin_amdgcn_sched_barrier(0);
	typename Mfma<float>::acc_t acc;
	#pragma unroll
	for (int r = 0; r < 16; ++r)
		acc[r] = 0.f;
	const bool sums_bias = kt == 0 && bgrad != nullptr;
	float bias[LOADS];
	#pragma unroll
	for (int q = 0; q < LOADS; ++q)
		bias[q] = 0.f;
	f32x4* const xs = stage + wave * 2 * GL * UNITS;
	f32x4* const zs = xs + GL * UNITS;
	#pragma unroll
	for (int h = 0; h < HALVES; ++h) {
		if constexpr (ACT) {
			#pragma unroll
			for (int q = 0; q < LOADS; ++q)
				#pragma unroll
				for (int i = 0; i < 4; ++i)
					gv[h][q][i] = (sign_bit(yv[h][q][i]) ? p1 * yv[h][q][i] + p0 : 1.f) * gv[h][q][i];
			if (act_dz != nullptr && kt == 0 && m0 + h * HALF_M < M) {
				#pragma unroll
				for (int q = 0; q < LOADS; ++q)
					if (f0 + row + ROWS * q < F)
						__builtin_nontemporal_store(gv[h][q], reinterpret_cast<f32x4*>(act_dz + ((size_t) M * (f0 + row + ROWS * q) + m0 + h * HALF_M)));
			}
		}
		#pragma unroll
		for (int q = 0; q < LOADS; ++q) {
			zs[unit_of(row + ROWS * q, unit)] = gv[h][q];
			xs[unit_of(row + ROWS * q, unit)] = xv[h][q];
			#pragma unroll
			for (int i = 0; i < 4; ++i)
				bias[q] += gv[h][q][i];
		}
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
	float* const part = reinterpret_cast<float*>(xs);
	#pragma unroll
	for (int r = 0; r < 16; ++r)
		part[acc_row<float>(r, lk) * GL + lc] = acc[r];
	if (sums_bias) {
		#pragma unroll
		for (int q = 0; q < LOADS; ++q) {
			#pragma unroll
			for (int off = 1; off < UNITS; off *= 2)
				bias[q] += __shfl_xor(bias[q], off, 64);
			if (unit == 0)
				part[GL * GL + row + ROWS * q] = bias[q];
		}
	}
	__syncthreads();
	constexpr int STRIDE = 2 * GL * GL;
	const float* const red = reinterpret_cast<const float*>(stage);
	const auto add = [&](int o, float old, bool fetched) {
		float v = red[o];
		for (int w = 1; w < waves; ++w)
			v += red[w * STRIDE + o];
		const int k = k0 + o % GL, f = f0 + o / GL;
		if (k < K && f < F) {
			float* dst = wgrad + ((size_t) k + (size_t) K * f);
			*dst = (fetched ? old : fresh ? 0.f : *dst) + v;
		}
	};
	#pragma unroll
	for (int i = 0; i < 4; ++i)
		if (tid + i * (int) blockDim.x < GL * GL)
			add(tid + i * (int) blockDim.x, before[i], true);
	for (int o = tid + 4 * (int) blockDim.x; o < GL * GL; o += blockDim.x)
		add(o, 0.f, false);
	if (sums_bias && tid < GL && f0 + tid < F) {
		float v = red[GL * GL + tid];
		for (int w = 1; w < waves; ++w)
			v += red[w * STRIDE + GL * GL + tid];
		bgrad[f0 + tid] = fresh ? v : bgrad[f0 + tid] + v;
	}
}

bool is_dense(const GatherGeom& g) {
	return g.R == 1 && g.S == 1 && g.LH == 1 && g.LW == 1 && g.OA == 1 && g.OB == 1 && g.N == g.NS && g.M == g.N && g.K == g.LC &&
			g.PA == 0 && g.PB == 0 && g.DA == 1 && g.DB == 1 && g.out_M == g.M && g.out_a0 == 0 && g.out_b0 == 0 && g.out_sa == 1 && g.out_sb == 1;
}
int up(int n, int d) {
	return (n + d - 1) / d;
}

} /* namespace */

bool addressable_product(const GatherGeom& g) {
	return is_dense(g) && 4.0 * g.M * (g.K + 64.0) < 2147483648.0 && 4.0 * (g.K + 64.0) * g.ldw < 2147483648.0;
}
bool small_product_possible(const GatherGeom& g, int cus) {
	if (!addressable_product(g))
		return false;
	/* Up to two tiles per CU, three where the reduction is short; more tiles, and reductions of more than three batches of loads a
	 * wavefront, go to the tiled launches. Whole passes, this kernel against those: 256 x 3072 -> 128 32.6 us against 45.4, 512 x 600
	 * x 600 (608 tiles) 41.6 / 48.1, 256 x 512 x 1500 (752) 33.7 / 36.1; but 128 x 2048 x 3000 (752) 89.4 / 86.3, 2048 x 500 x 200 (832) 44.1 /
	 * 43.0, and 128 x 8192 -> 256 66.3 / 57.6 (at 5000 inputs as fast). Below 32 reduction indices there is nothing to deal out. Forward
	 * launches of few columns, this kernel against those: 128 x 1100 -> 10 4.8 / 7.3, 128 x 3072 -> 10 8.3 / 10.4, 1 x 2000 -> 10 7.0 / 12.4,
	 * 128 x 2000 -> 2 6.2 / 53.9 (few_columns_plain_kernel). */
	const long tiles = (long) up(g.M, 2 * PL) * up(g.F, PL);
	return g.K >= 32 && g.K <= 3072 && tiles <= (g.K <= 1024 ? 3 : 2) * (long) cus;
}

namespace {
ProductArgs product_args(const GatherGeom& g, int wt_rows, const Epilogue<float>* E, int rows, int columns) {
	ProductArgs A;
	A.M = g.M; A.K = g.K; A.F = g.F; A.ldw = g.ldw;
	A.mtiles = up(g.M, rows);
	A.tiles = A.mtiles * up(g.F, columns);
	A.x_bytes = 4u * (unsigned) g.M * (unsigned) g.K;
	A.wt_bytes = 4u * (unsigned) wt_rows * (unsigned) g.ldw;
	A.kind = E ? E->kind : -1;
	A.p = E ? E->p : 0.f;
	A.pre = E ? E->pre : nullptr;
	return A;
}
} /* namespace */

void small_product_ordered(const float* src, const float* wt, const float* bias, float* out, const GatherGeom& g, int wt_rows,
		const Epilogue<float>* E, int waves) {
	ProductArgs A = product_args(g, wt_rows, E, OL, OL);
	A.per = up(g.K / OK, waves);
	small_product_ordered_kernel<<<dim3((unsigned) up(A.tiles, 8) * 8), dim3(64u * (unsigned) waves), 0, stream()>>>(src, wt, bias, out, A);
	CATTLE_HIP_CHECK(hipGetLastError());
}

void small_product(const float* src, const float* wt, const float* bias, float* out, const GatherGeom& g, int wt_rows,
		const Epilogue<float>* E, int cus) {
	/* 32 rows per block where that gives every CU one, else 16; 16 too where the reduction is long, which takes more accumulators */
	const int mb = up(g.M, 2 * PL) * up(g.F, PL) >= cus && g.K <= 1536 ? 2 : 1;
	const bool pairs = mb == 2 && g.M % 2 == 0 && (reinterpret_cast<uintptr_t>(src) & 7) == 0;
	ProductArgs A = product_args(g, wt_rows, E, PL * mb, PL);
	const int steps = up(g.K, PK), most = A.tiles <= cus || g.K > 1536 ? 16 : 8;
	A.per = up(steps, most);
	const dim3 grid((unsigned) up(A.tiles, 8) * 8), block(64u * (unsigned) up(steps, A.per));
	const auto launch = [&](auto tail) {
		constexpr bool TAIL = decltype(tail)::value;
		if (pairs)
			small_product_kernel<2, true, TAIL><<<grid, block, 0, stream()>>>(src, wt, bias, out, A);
		else if (mb == 2)
			small_product_kernel<2, false, TAIL><<<grid, block, 0, stream()>>>(src, wt, bias, out, A);
		else
			small_product_kernel<1, false, TAIL><<<grid, block, 0, stream()>>>(src, wt, bias, out, A);
	};
	g.K % PK == 0 ? launch(std::false_type()) : launch(std::true_type());
	CATTLE_HIP_CHECK(hipGetLastError());
}

bool small_weight_gradient_possible(const GatherGeom& g, bool vec, const WgradAct<float>* act) {
	return is_dense(g) && vec && (act == nullptr || act->pool_inds == nullptr) && g.M <= 2 * HALF_M * GRAD_WAVES && g.F >= GL &&
			4.0 * g.M * std::max(g.K, g.F) < 1073741824.0;
}

void small_weight_gradient(const float* x, const float* og, float* wgrad, float* bgrad, const GatherGeom& g, const WgradAct<float>* act,
		float p0, float p1, bool fresh) {
	const int ktiles = up(g.K, GL), tiles = ktiles * up(g.F, GL);
	/* 32 samples a wavefront where eight wavefronts hold the batch and the tiles are few, else 64: 256 x 784 x 512 (400 tiles) 8.1 -> 7.7 us,
	 * a pass of that MLP 427 -> 422; but the pass of one with 3072 tiles 403 -> 427, whose blocks fill the chip either way and have twice
	 * as many partial tiles to add. */
	const int halves = g.M <= HALF_M * GRAD_WAVES && tiles <= 512 ? 1 : 2;
	const dim3 grid((unsigned) up(tiles, 8) * 8), block(64u * (unsigned) up(g.M, halves * HALF_M));
	const unsigned x_bytes = 4u * (unsigned) g.M * (unsigned) g.K, og_bytes = 4u * (unsigned) g.M * (unsigned) g.F;
	const size_t lds = (block.x / 64) * 2 * GL * GL * sizeof(float);
	const auto launch = [&](auto undoes, auto h) {
		small_weight_gradient_kernel<decltype(undoes)::value, decltype(h)::value><<<grid, block, lds, stream()>>>(x, og, wgrad, bgrad, g.M, g.K, g.F,
				ktiles, tiles, x_bytes, og_bytes, act ? act->y : nullptr, act ? act->dz : nullptr, p0, p1, fresh);
	};
	typedef std::integral_constant<int, 1> one;
	typedef std::integral_constant<int, 2> two;
	if (act)
		halves == 1 ? launch(std::true_type(), one()) : launch(std::true_type(), two());
	else
		halves == 1 ? launch(std::false_type(), one()) : launch(std::false_type(), two());
	CATTLE_HIP_CHECK(hipGetLastError());
}

} /* namespace cattle_hip */
