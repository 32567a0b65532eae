/*
 * lstm_steps.hip — a time step of a 3 x 3 convolutional LSTM cell as one launch: the recurrent product on the fp32 matrix
 * instructions and the element-wise part of the step on its sums.
 */
#include "lstm_steps.hpp"
#include "lstm_math.hpp"
#include "tap_product.hpp"

namespace cattle_hip {
namespace {

using namespace tap_product;

/* What a step reads of the state arrives before the product's loads are issued. With both in flight at once a step of 8192 x 288 x 128
 * takes 15.9 us forward and 15.1 backward under the profiler, in this order 12.4 and 11.7; a pass of 10 time steps in both directions 397 and
 * 337 us. (Waits for vector memory only: 0 of its counter, the others left alone.) */
__device__ __forceinline__ void wait_for_state() {
	__builtin_amdgcn_s_waitcnt(0x0F70);
	__builtin_amdgcn_sched_barrier(0);
}

/* Forward step t: the weighted previous output of the four gates, then gates, state and hidden output. A block owns 32 rows
 * (samples and positions) and up to four groups of eight hidden channels; a wavefront a group's 32 columns, eight channels for
 * each of the four gates, and a quarter of the source channels. The four partial tiles of a group meet in LDS, and a thread
 * adds the sums of one state element, in ascending order, and runs its step; what the step reads besides is fetched first.
 * Bound by latency and the fp32 matrix instructions, 3.9 us of them for 8192 x 288 x 128 on 256 blocks: there 17.0 us under the
 * profiler as 64 x 64 tiles of gather_gemm_kernel (EPI_LSTM), whose five chunks of the reduction were five round trips to memory, and
 * 11.9 here. (Without its products 9.5, without most of its loads 9.9, with neither 6.3, of which an empty launch is 4.7.) */
template<int SPC>
__global__ __launch_bounds__(1024)
void lstm_step_forward_kernel(const float* __restrict__ src, const float* __restrict__ wt, const float* __restrict__ bias,
		const GatherGeom g, const StepGeom G, const LstmForwardStep<float> A) {
	constexpr int SPLITS = 4, CB = LSTM_STEP_GATE_BLOCK;
	extern __shared__ float red[];                  /* [split][group][column][row] */
	const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
	const int groups = blockDim.x / (64 * SPLITS), group0 = (int) blockIdx.y * groups;
	const int hidden = g.F / 4, split = wave % SPLITS, group = wave / SPLITS;
	const int lc = lane % TL, lk = lane / TL;
	const unsigned m = blockIdx.x * TL + (unsigned) lc;
	const bool valid = (int) m < g.M;
	const Row row = row_of(valid ? m : 0u, g, G);

	/* thread tid: row lc of the tile, hidden channel tid / 32 of the block's */
	const int h = group0 * CB + tid / TL;
	const bool mine = valid && h < hidden;
	const unsigned positions = (unsigned) (g.OA * g.OB), rest = row.pos + positions * (unsigned) (mine ? h : 0);
	const unsigned e = row.n + (unsigned) g.N * rest, slab_rows = positions * (unsigned) hidden;
	const LstmForwardInputs<float> in = lstm_forward_load_at<float>(A, e, row.n, rest, slab_rows);
	float bv[4];
	#pragma unroll
	for (int q = 0; q < 4; ++q)
		bv[q] = bias ? bias[q * hidden + (mine ? h : 0)] : 0.f;
	wait_for_state();

	if ((group0 + group) * CB < hidden) {           /* (the same for the whole wavefront) */
		const acc_t acc = share_of_product<SPC>(src, wt, g, G, row, valid, lk, (group0 + group) * 4 * CB + lc, split * 2 * SPC);
		float* dst = red + (split * groups + group) * TL * TL + lc;
		#pragma unroll
		for (int r = 0; r < 16; ++r)
			dst[acc_row<float>(r, lk) * TL] = acc[r];
	}
	__syncthreads();
	if (!mine)
		return;
	const int j = tid / TL;
	const float* col = red + ((j / CB) * TL + j % CB) * TL + lc;
	float zh[4];
	#pragma unroll
	for (int q = 0; q < 4; ++q) {
		zh[q] = col[q * CB * TL];
		#pragma unroll
		for (int s = 1; s < SPLITS; ++s)
			zh[q] += col[(s * groups * TL + q * CB) * TL];
		zh[q] += bv[q];
	}
	if (lstm_standard_acts(A.a))
		lstm_forward_store_at<float>(A, e, row.n, rest, lstm_forward_compute<float, true>(A, in, true, zh));
	else
		lstm_forward_store_at<float>(A, e, row.n, rest, lstm_forward_compute<float, false>(A, in, true, zh));
}

/* Backward step: the gradient of the hidden output that comes back through the recurrent kernels of the step after, and on it
 * the step's element-wise backward pass. A block owns 32 rows and 32 hidden channels, each of its sixteen wavefronts a
 * sixteenth of the source channels. Bound as the forward step: 8192 x 1152 x 32 took 13.5 us under the profiler as
 * wave_split_gemm_kernel, whose wavefronts wait for memory two or three times, and 11.4 here. */
template<int SPC>
__global__ __launch_bounds__(1024)
void lstm_step_backward_kernel(const float* __restrict__ src, const float* __restrict__ wt, const GatherGeom g, const StepGeom G,
		const LstmBackwardStep<float> A) {
	constexpr int SPLITS = 16;
	__shared__ float red[SPLITS * TL * TL];         /* [split][column][row] */
	const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
	const int lc = lane % TL, lk = lane / TL, f0 = (int) blockIdx.y * TL;
	const unsigned m = blockIdx.x * TL + (unsigned) lc;
	const bool valid = (int) m < g.M;
	const Row row = row_of(valid ? m : 0u, g, G);

	const int h = f0 + tid / TL;
	const bool mine = valid && h < g.F;
	const unsigned positions = (unsigned) (g.OA * g.OB), rest = row.pos + positions * (unsigned) (mine ? h : 0);
	const unsigned e = row.n + (unsigned) g.N * rest, slab_rows = positions * (unsigned) g.F;
	const LstmBackwardInputs<float> in = lstm_backward_load_at<float>(A, e, row.n, rest, true);
	wait_for_state();

	const acc_t acc = share_of_product<SPC>(src, wt, g, G, row, valid, lk, f0 + lc, wave * 2 * SPC);
	float* dst = red + wave * TL * TL + lc;
	#pragma unroll
	for (int r = 0; r < 16; ++r)
		dst[acc_row<float>(r, lk) * TL] = acc[r];
	__syncthreads();
	if (!mine)
		return;
	float dh = red[tid];
	#pragma unroll
	for (int s = 1; s < SPLITS; ++s)
		dh += red[s * TL * TL + tid];
	if (lstm_standard_acts(A.a))
		lstm_backward_finish_at<float, true>(A, e, row.n, rest, slab_rows, true, dh, in);
	else
		lstm_backward_finish_at<float, false>(A, e, row.n, rest, slab_rows, true, dh, in);
}

/* At most six row tiles per CU. A CU holds one block of these kernels, whose waits overlap with nothing of another's, while the
 * launches over many rows keep the matrix pipes busy. A training pass over 4 steps, the step kernels against those launches,
 * at 4.5 tiles per CU: 525 us against 629 (32 hidden channels); at 8: 233 against 328 (8), 400 against 462 (16), but 807 against 807
 * (32) and 1633 against 1609 (48). */
bool few_rounds(int M, int cus) {
	return tiles_of(M) <= 6 * cus;
}

template<typename Fn>
void with_steps(int spc, Fn fn) {
	switch (spc) {
	case 1: fn(std::integral_constant<int, 1>()); break;
	case 2: fn(std::integral_constant<int, 2>()); break;
	case 3: fn(std::integral_constant<int, 3>()); break;
	case 4: fn(std::integral_constant<int, 4>()); break;
	case 5: fn(std::integral_constant<int, 5>()); break;
	default: fn(std::integral_constant<int, 6>());
	}
}

} /* namespace */

bool lstm_step_forward_possible(const GatherGeom& g, const LstmForwardStep<float>& step, int cus) {
	return addressable(g) && g.F == 4 * g.LC && g.LC % 8 == 0 && g.LC <= 48 && step.P == (size_t) g.M * g.LC && few_rounds(g.M, cus) &&
			g.N % 4 == 0;
}
bool lstm_step_backward_possible(const GatherGeom& g, const LstmBackwardStep<float>& step, int cus) {
	return addressable(g) && g.LC == 4 * g.F && g.F % 8 == 0 && g.F <= 48 && step.P == (size_t) g.M * g.F && step.z == nullptr &&
			step.zx_fwd == nullptr && few_rounds(g.M, cus);
}

void lstm_step_forward(const float* src, const float* wt, const float* bias, const GatherGeom& g, const LstmForwardStep<float>& step) {
	constexpr int SPLITS = 4;
	/* as many groups per block as divide them evenly, at most four (1024 threads) */
	const int groups = g.LC / LSTM_STEP_GATE_BLOCK, blocks_f = (groups + 3) / 4, per_block = (groups + blocks_f - 1) / blocks_f;
	const dim3 grid((unsigned) tiles_of(g.M), (unsigned) blocks_f), block(64u * SPLITS * (unsigned) per_block);
	const size_t lds = sizeof(float) * SPLITS * per_block * TL * TL;
	const StepGeom G = step_geom(g);
	with_steps(g.LC / 8, [&](auto spc) {
		lstm_step_forward_kernel<decltype(spc)::value><<<grid, block, lds, stream()>>>(src, wt, bias, g, G, step);
	});
	CATTLE_HIP_CHECK(hipGetLastError());
}

void lstm_step_backward(const float* src, const float* wt, const GatherGeom& g, const LstmBackwardStep<float>& step) {
	const dim3 grid((unsigned) tiles_of(g.M), (unsigned) tiles_of(g.F));
	const StepGeom G = step_geom(g);
	with_steps(g.F / 8, [&](auto spc) {
		lstm_step_backward_kernel<decltype(spc)::value><<<grid, 1024, 0, stream()>>>(src, wt, g, G, step);
	});
	CATTLE_HIP_CHECK(hipGetLastError());
}

} /* namespace cattle_hip */
