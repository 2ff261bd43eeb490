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

// Piece `item` when the runs of more than `at_most` tokens are cut into pieces of `tokens`, in order: tokens in it (0: there is no
// such piece), its sequence, the run's tokens in front of it and the chunks of the runs before.  Every lane of a wave calls.
__device__ __forceinline__ int lw_find_piece(const int32_t* __restrict__ q_start, int num_seqs, int at_most, int tokens, int item,
                                             int* seq, int* tok0, int* chunks_before) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  if (num_seqs <= 8) {                           // (the lanes' sums take a microsecond a call)
    for (int s = 0; s < num_seqs; ++s) {
      int n = q_start[s + 1] - q_start[s];
      n = n > at_most ? n : 0;
      const int pieces = (n + tokens - 1) / tokens;
      if (item < pieces) {
        *seq = s;
        *tok0 = item * tokens;
        *chunks_before = before;
        return n - *tok0 < tokens ? n - *tok0 : tokens;
      }
      item -= pieces;
      before += (n + kLwChunk - 1) / kLwChunk;
    }
    return 0;
  }
  for (int s0 = 0; s0 < num_seqs; s0 += 64) {
    const int s = s0 + lane;
    int n = s < num_seqs ? q_start[s + 1] - q_start[s] : 0;
    n = n > at_most ? n : 0;
    const int pieces = (n + tokens - 1) / tokens, chunks = (n + kLwChunk - 1) / kLwChunk;
    int upto = pieces, cupto = chunks;           // of the sequences up to this lane's
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const int a = __shfl_up(upto, m, 64), b = __shfl_up(cupto, m, 64);
      if (lane >= m) upto += a, cupto += b;
    }
    const uint64_t past = __builtin_amdgcn_ballot_w64(upto > item);
    if (past != 0) {
      const int l = __builtin_ctzll(past);
      const int t0 = (item - __builtin_amdgcn_readlane(upto - pieces, l)) * tokens;
      *seq = s0 + l;
      *tok0 = t0;
      *chunks_before = before + __builtin_amdgcn_readlane(cupto - chunks, l);
      const int left = __builtin_amdgcn_readlane(n, l) - t0;
      return left < tokens ? left : tokens;
    }
    item -= __builtin_amdgcn_readlane(upto, 63);
    before += __builtin_amdgcn_readlane(cupto, 63);
  }
  return 0;
}

// S <- diag(a_t) S + k v^T with a_t = sigmoid(decay_pre + bias)^(1 / tau) per key channel, o = S^T (q_scale q)
int gla_walk(const LinearStep& a, const LinearWalkPlan& plan, const void* decay_pre, int64_t decay_stride, const float* decay_bias, float inv_tau, float q_scale,
             int act_dtype, hipStream_t stream);
// S <- decay_h S + k v^T, o = S^T q; silu: q, k and v pass a silu first.  q and k in q_dtype, v in v_dtype.
int lightning_walk(const LinearStep& a, const LinearWalkPlan& plan, const float* decay, bool silu, int q_dtype, int v_dtype, hipStream_t stream);

}  // namespace swm
