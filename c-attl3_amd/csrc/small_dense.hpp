/*
 * small_dense.hpp — launch interface of the kernels for fp32 matrix products of a dense layer that are too small to fill the chip
 * with tiles (small_dense.hip).
 */
#ifndef CATTLE_HIP_SMALL_DENSE_HPP_
#define CATTLE_HIP_SMALL_DENSE_HPP_

#include "gemm_tiles.hpp"

namespace cattle_hip {

/* Whether the product src[M x K] wt[K x F] of this gather is one of small_product's: no positions, no output map, few tiles. */
bool small_product_possible(const GatherGeom& g, int cus);
/* out = src wt + bias, with an activation (E, EPI_ACT) if E is given; wt: prepared weights of wt_rows rows (zeros past g.K). Any
 * batch size and alignment. */
void small_product(const float* src, const float* wt, const float* bias, float* out, const GatherGeom& g, int wt_rows,
		const Epilogue<float>* E, int cus);
/* The same with its sums taken as wave_split_gemm_kernel takes them with `waves` wavefronts (addressable_product, g.K even). */
bool addressable_product(const GatherGeom& g);
void small_product_ordered(const float* src, const float* wt, const float* bias, float* out, const GatherGeom& g, int wt_rows,
		const Epilogue<float>* E, int waves);

/* Whether the weight gradient of a dense layer (g: its forward gather) is one of small_weight_gradient's; x, the gradient and
 * what `act` holds lie on 16-byte boundaries and g.N is a multiple of four (`vec`). */
bool small_weight_gradient_possible(const GatherGeom& g, bool vec, const WgradAct<float>* act);
/* wgrad += x^T z, bgrad += column sums of z, with z the gradient og or, with `act`, what WgradAct says (p0 + p1 y: the derivative
 * on the negative side); with `fresh` the gradients are overwritten, not added to */
void small_weight_gradient(const float* x, const float* og, float* wgrad, float* bgrad, const GatherGeom& g, const WgradAct<float>* act,
		float p0, float p1, bool fresh);

} /* namespace cattle_hip */

#endif /* CATTLE_HIP_SMALL_DENSE_HPP_ */
