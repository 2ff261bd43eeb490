// delta_step.hip: short runs of the delta rule in one launch
#pragma once

#include <stdint.h>

#include <hip/hip_runtime.h>

namespace swm {

// The step's sequences of at most `at_most` tokens; false when the sizes or addresses are not for it, and then nothing was done.
bool delta_step(float* out, const float* qkv, const void* beta_pre, int64_t beta_stride, const void* decay_pre,
                int64_t decay_stride, int decay_per_head, const float* dt_bias, const float* a_log, float* state,
                const int32_t* q_start, const int32_t* ctx_len, const int32_t* state_slot, int num_seqs, int heads, int kv_heads,
                int dim, int vdim, int at_most, int act_dtype, hipStream_t stream);

}  // namespace swm
