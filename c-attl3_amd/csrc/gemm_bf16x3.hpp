/*
 * gemm_bf16x3.hpp — launch interface of the fp32 GEMM kernels that multiply on the bf16 matrix instructions
 * (gemm_bf16x3.hip).
 */
#ifndef CATTLE_HIP_GEMM_BF16X3_HPP_
#define CATTLE_HIP_GEMM_BF16X3_HPP_

#include "gemm_tiles.hpp"

namespace cattle_hip {

/* Tile shapes of gather_gemm_bf16x3_kernel: rows, columns and wavefronts of a block. */
struct Bf16x3Tile { int bm, bf, waves, lds_bytes; };
constexpr int BF16X3_KC = 32;           /* reduction chunk of every shape */
constexpr int BF16X3_TILES = 5;
enum { BF16X3_256x128 = 0, BF16X3_256x64 = 1, BF16X3_128x64 = 2, BF16X3_64x64 = 3, BF16X3_128x32 = 4 };
Bf16x3Tile bf16x3_tile(int shape);
/* Whether the kernel can address the problem: no divisors, at most 31 taps, operands of less than 2^31 bytes. */
bool bf16x3_gather_possible(const GatherGeom& g);
/* wt: the prepared fp32 weights; wt_rows their padded row count. epi: EPI_NONE, or EPI_ACT, EPI_POOL, EPI_STATS where the
 * batch is a multiple of four and src and out lie on 16-byte boundaries. */
void bf16x3_gather(int shape, const float* src, const float* wt, const float* bias, float* out, const GatherGeom& g,
		const GatherLaunch& L, float* partials, int wt_rows, int epi, const Epilogue<float>& E);
/* the problems of a table in one launch: N even, src on an 8-byte boundary (pairs of samples), no bias, weights padded to
 * wt_row_pad rows */
void bf16x3_gather_classes(int shape, int classes_used, const float* src, float* out, const GatherClasses<float>& classes, int wt_row_pad);
int bf16x3_gather_blocks_per_cu(int shape);

/* Tile shapes of wgrad_bf16x3_kernel (K rows x F columns): 192 x 128, 96 x 128, 128 x 64, 64 x 64. */
constexpr int BF16X3_WGRAD_TILES = 4;
struct Bf16x3WgradPlan {
	int shape;
	int ktiles, tiles, splits, chunks_per_split;
	int pixels;             /* slices are ranges of output positions (N % 32 == 0 and 16-byte boundaries), else of chunks of 32 rows */
	int direct;             /* one slice: the block adds its tile to the gradient itself */
};
void bf16x3_wgrad_tile(int shape, int* bk, int* bf);
int bf16x3_wgrad_blocks_per_cu(int shape);
bool bf16x3_wgrad_possible(const GatherGeom& g);
void bf16x3_wgrad(const Bf16x3WgradPlan& plan, const float* src, const float* og, float* partials, float* bias_partials, const GatherGeom& g);

} /* namespace cattle_hip */

#endif /* CATTLE_HIP_GEMM_BF16X3_HPP_ */
