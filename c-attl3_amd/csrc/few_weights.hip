/*
 * few_weights.hip — the launch of few_weights.hpp's weight gradient.
 */
#include "few_weights.hpp"

namespace cattle_hip {
namespace {

using namespace few_weights;

/* grid = (slices, tiles of 32 weights) */
template<int GQ>
__global__ __launch_bounds__(64 * WAVES)
void few_weights_kernel(const FewWeights A) {
	extern __shared__ f32x4 few_weights_stage[];
	few_weights_body<GQ>(A, (int) blockIdx.x, (int) blockIdx.y, few_weights_stage);
}

int groups_of(const GatherGeom& g) {
	return (g.N + ITEM - 1) / ITEM;
}
int items_of(const GatherGeom& g) {
	return g.M / g.N * groups_of(g);
}

} /* namespace */

bool few_weights_possible(const GatherGeom& g, bool vec) {
	return vec && g.K <= 2 * TL && g.F <= 16 && g.DA == 1 && g.DB == 1 && g.N == g.NS && g.M / g.N >= 16 &&
			4.0 * g.NS * g.LH * g.LW * g.LC < 2147483648.0 && 4.0 * g.M * g.F < 2147483648.0;
}

int few_weights_slices(const GatherGeom& g, int most) {
	/* a wavefront per item, four to a block, where that many slices may be written */
	const int items = items_of(g), slices = std::min(most, (items + 3) / 4);
	const int per = (items + slices - 1) / slices;
	return (items + per - 1) / per;
}

few_weights::FewWeights few_weights_problem(const float* x, const float* og, float* partials, float* bias_partials, const GatherGeom& g, int slices,
		bool transposed) {
	const int items = items_of(g), per = (items + slices - 1) / slices;
	return { x, og, partials, bias_partials, g, items, groups_of(g), per, slices, transposed, 4u * (unsigned) (g.NS * g.LH * g.LW) * (unsigned) g.LC,
			4u * (unsigned) g.M * (unsigned) g.F };
}

void few_weights_gradient(const few_weights::FewWeights& A) {
	const int waves = std::min(A.per_slice, WAVES);
	const dim3 grid((unsigned) A.slices, (unsigned) ((A.g.K + TL - 1) / TL)), block(64u * (unsigned) waves);
	const size_t lds = (size_t) waves * 2 * TL * TL * sizeof(float);
	if (A.g.F <= 8)
		few_weights_kernel<1><<<grid, block, lds, stream()>>>(A);
	else
		few_weights_kernel<2><<<grid, block, lds, stream()>>>(A);
	CATTLE_HIP_CHECK(hipGetLastError());
}

} /* namespace cattle_hip */
