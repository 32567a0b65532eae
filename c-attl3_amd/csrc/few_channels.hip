/*
 * few_channels.hip — the fp32 3 x 3 convolution of up to six channels: products with so short a reduction that a wavefront
 * fetches all of its operands at once.
 */
#include "few_channels.hpp"
#include "tap_product.hpp"

namespace cattle_hip {
namespace {

using namespace tap_product;

/* A wavefront owns 32 rows and 32 columns and the whole reduction; nothing is staged, and the wavefronts of a CU cover each other's
 * waits. The wavefronts of a block are the column tiles of the same rows, or neighbouring rows: what they share comes from the
 * caches. gather_gemm_kernel takes such a reduction in two to seven chunks with a barrier and a round trip to memory each:
 * 65,536 x 27 x 16 7.7 -> 6.2 us. Bound by latency. */
template<int SPC, bool ODD>
__global__ __launch_bounds__(256)
void few_channels_kernel(const float* __restrict__ src, const float* __restrict__ wt, const float* __restrict__ bias, float* __restrict__ out,
		const GatherGeom g, const StepGeom G, int ftiles, int tiles, int blocks) {
	const int block = xcd_tile(blockIdx.x, blocks);
	const int lane = threadIdx.x % 64, tile = block * 4 + __builtin_amdgcn_readfirstlane((int) threadIdx.x / 64);
	if (block >= blocks || tile >= tiles)
		return;
	const int mt = tile / ftiles, f0 = (tile - mt * ftiles) * TL;
	const int lc = lane % TL, lk = lane / TL;
	const unsigned m = (unsigned) (mt * TL + lc);
	const bool valid = (int) m < g.M;
	const Row row = row_of(valid ? m : 0u, g, G);
	float bv[16];
	#pragma unroll
	for (int r = 0; r < 16; ++r)
		bv[r] = bias != nullptr ? bias[min(f0 + acc_row<float>(r, lk), g.F - 1)] : 0.f;
	const acc_t acc = share_of_product<SPC, ODD>(src, wt, g, G, row, valid, lk, f0 + lc, 0);
	if (!valid)
		return;
	#pragma unroll
	for (int r = 0; r < 16; ++r) {
		const int f = f0 + acc_row<float>(r, lk);
		if (f < g.F)
			__builtin_nontemporal_store(acc[r] + bv[r], out + ((size_t) m + (size_t) g.M * f));
	}
}

} /* namespace */

bool few_channels_possible(const GatherGeom& g, int cus) {
	/* Up to eight wavefronts of 32 x 32 per CU. More of them are better served by tiles that are fetched once for
	 * several: a pass of 524,288 x 27 x 16 85 us against 74.5, one of 81,920 x 72 x 128 42 us against 27; and longer reductions by the
	 * chunks that overlap the products (3200 x 108 x 64 28.0 against 27.1). 25,088 x 54 x 10 27.2 against 31.9. */
	const double tiles = (double) tiles_of(g.M) * tiles_of(g.F);
	return addressable(g) && g.LC <= 6 && tiles <= 8.0 * cus && g.F > 8 && g.out_M == g.M && g.out_a0 == 0 && g.out_b0 == 0 && g.out_sa == 1 && g.out_sb == 1 &&
			g.out_OA == g.OA;
}

void few_channels_product(const float* src, const float* wt, const float* bias, float* out, const GatherGeom& g) {
	const int ftiles = tiles_of(g.F), tiles = tiles_of(g.M) * ftiles, blocks = (tiles + 3) / 4;
	const StepGeom G = step_geom(g);
	const dim3 grid((unsigned) ((blocks + 7) / 8 * 8));
	switch (g.LC) {
#define CATTLE_HIP_CHANNELS(n) case n: few_channels_kernel<(n + 1) / 2, n % 2 != 0><<<grid, 256, 0, stream()>>>(src, wt, bias, out, g, G, ftiles, tiles, blocks); break;
	CATTLE_HIP_CHANNELS(1) CATTLE_HIP_CHANNELS(2) CATTLE_HIP_CHANNELS(3) CATTLE_HIP_CHANNELS(4) CATTLE_HIP_CHANNELS(5) CATTLE_HIP_CHANNELS(6)
#undef CATTLE_HIP_CHANNELS
	}
	CATTLE_HIP_CHECK(hipGetLastError());
}

} /* namespace cattle_hip */
