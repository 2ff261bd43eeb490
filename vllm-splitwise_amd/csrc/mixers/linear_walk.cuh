// Long runs of the linear-attention rules (linear_walk.hip): arguments shared with gla.hip and lightning.hip.
#pragma once

#include "linear_plan.h"
#include "mixers_common.cuh"

namespace swm {

struct LinearStep {
  float* out;
  const void *q, *k, *v;
  int64_t qk_stride, v_stride;          // elements between rows
  float* state;
  const int32_t *q_start, *ctx_len, *state_slot;
  int64_t rows;
  int num_seqs, heads, dim, vdim;
  float* workspace;
};

// S <- diag(a_t) S + k v^T with a_t = sigmoid(decay_pre + bias)^(1 / tau) per key channel, o = S^T (q_scale q)
int gla_walk(const LinearStep& a, const LinearWalkPlan& plan, const void* decay_pre, int64_t decay_stride, const float* decay_bias, float inv_tau, float q_scale,
             int act_dtype, hipStream_t stream);
// S <- decay_h S + k v^T, o = S^T q; silu: q, k and v pass a silu first.  q and k in q_dtype, v in v_dtype.
int lightning_walk(const LinearStep& a, const LinearWalkPlan& plan, const float* decay, bool silu, int q_dtype, int v_dtype, hipStream_t stream);

// The same token by token for sequences of at most `at_most` tokens, in linear_step.hip (-> false: not in this form)
bool gla_step(const LinearStep& a, const void* decay_pre, int64_t decay_stride, const float* decay_bias, float inv_tau, float q_scale,
              int at_most, int act_dtype, hipStream_t stream);
bool lightning_step(const LinearStep& a, const float* decay, bool silu, int at_most, int v_dtype, hipStream_t stream);

}  // namespace swm
