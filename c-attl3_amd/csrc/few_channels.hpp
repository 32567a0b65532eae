/*
 * few_channels.hpp — launch interface of the fp32 3 x 3 convolution of a few channels (few_channels.hip).
 */
#ifndef CATTLE_HIP_FEW_CHANNELS_HPP_
#define CATTLE_HIP_FEW_CHANNELS_HPP_

#include "gemm_tiles.hpp"

namespace cattle_hip {

/* Whether the product of this gather is one of few_channels_product's: 3 x 3 taps without divisors, a handful of channels, the plain
 * output map, on a chip of `cus` CUs. */
bool few_channels_possible(const GatherGeom& g, int cus);
/* out = gather(src) wt + bias; any batch size and alignment */
void few_channels_product(const float* src, const float* wt, const float* bias, float* out, const GatherGeom& g);

} /* namespace cattle_hip */

#endif /* CATTLE_HIP_FEW_CHANNELS_HPP_ */
