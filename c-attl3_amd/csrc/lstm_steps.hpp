/*
 * lstm_steps.hpp — launch interface of the kernels that run one time step of a 3 x 3 convolutional LSTM cell, its recurrent
 * product and its element-wise part, as one launch (lstm_steps.hip).
 */
#ifndef CATTLE_HIP_LSTM_STEPS_HPP_
#define CATTLE_HIP_LSTM_STEPS_HPP_

#include "gemm_tiles.hpp"

namespace cattle_hip {

/* The gates of how many hidden channels stand together in the prepared weights of the forward step (lstm_gate_column) */
constexpr int LSTM_STEP_GATE_BLOCK = 8;
/* Whether the forward step, or the backward step, of this problem (the gather of its recurrent product) has such a kernel:
 * g.F = 4 * hidden columns forward; hidden columns and 4 * hidden channels backward, on a chip of `cus` CUs. */
bool lstm_step_forward_possible(const GatherGeom& g, const LstmForwardStep<float>& step, int cus);
bool lstm_step_backward_possible(const GatherGeom& g, const LstmBackwardStep<float>& step, int cus);
void lstm_step_forward(const float* src, const float* wt, const float* bias, const GatherGeom& g, const LstmForwardStep<float>& step);
void lstm_step_backward(const float* src, const float* wt, const GatherGeom& g, const LstmBackwardStep<float>& step);

} /* namespace cattle_hip */

#endif /* CATTLE_HIP_LSTM_STEPS_HPP_ */
