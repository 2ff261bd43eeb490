// Steps of capped_attention.hip that run on the bf16 matrix cores, prompts (prompt_attention.hip) and decode steps of few rows
// (decode_attention.hip): arguments.
#pragma once

#include "attention_plan.h"
#include "mixers_common.cuh"

namespace swm {

struct PromptAttention {
  void* out;
  const float* q;
  const uint16_t *key_cache, *value_cache, *gate;
  const int32_t *block_tables, *q_start, *ctx_len;
  const float *sink_logit, *score_bias;
  int64_t out_stride, gate_stride, k_stride, v_stride;
  int table_width, num_seqs, heads, kv_heads, dim, vdim, page_size, page_shift, window, chunk, sink, tpt;
  float scale, softcap;
};

// One query row over its keys in plain fp32, by one wave: what the matrix kernels fall back on for a row whose result is NaN.
// They take queries and weights apart into bf16 parts, and a part that is zero makes NaN of an infinity in the cache where the
// fp32 product is that infinity (a score of -inf hides its key, a capped score of inf is the cap, a value of inf stays one).
// q: the row's query; key_of(i), i < n: its keys, of which it sees those from `low` to `pos`; own: kPlainRowLds floats of LDS
// that are this wave's.  -> largest score, sum of weights (sigmoid weights: 0 and nothing) and the channels lane and lane + 64
// of the weighted values.  64 keys at a time, a lane each for the scores, the channels shared out for the values.
constexpr int kPlainRowLds = 128;
struct PlainRow {
  float m, l, o[2];
};
template <typename KeyOf>
__device__ __forceinline__ PlainRow plain_row(const PromptAttention& a, const int32_t* table, int g, const float* q, float bias,
                                              int pos, int low, int n, KeyOf key_of, float* own) {
  const int lane = threadIdx.x & 63;
  const bool sig = a.score_bias != nullptr;
  int page_size = a.page_size, dim = a.dim;
  asm volatile("" : "+s"(page_size), "+s"(dim));             // nothing of this in front of the branch to it
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  for (int c = lane; c < dim; c += 64) own[c] = q[c] * a.scale;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  PlainRow row{sig ? 0.0f : -INFINITY, 0.0f, {0.0f, 0.0f}};
  for (int i0 = 0; i0 < n; i0 += 64) {
    const int key = key_of(i0 + lane);
    const bool seen = i0 + lane < n && key <= pos && key >= low;
    const int slot = seen ? table[key / page_size] * page_size + key % page_size : 0;
    float s = 0.0f;
    if (seen) {
      const uint16_t* k = a.key_cache + (int64_t)slot * a.k_stride + (int64_t)g * a.dim;
      for (int c = 0; c < dim; ++c) s += own[c] * ld<bf16_t>(k, c);
    }
    if (a.softcap > 0.0f) s = a.softcap * fast_tanhf_(s / a.softcap);
    float p;
    if (sig) {
      p = seen ? __builtin_amdgcn_rcpf(1.0f + fast_expf_(-(s + bias))) : 0.0f;
    } else {
      if (!seen) s = -INFINITY;
      float most = s;
#pragma unroll
      for (int step = 32; step >= 1; step >>= 1) most = fmaxf(most, __shfl_xor(most, step, 64));
      const float m_new = fmaxf(row.m, most), m_use = m_new == -INFINITY ? 0.0f : m_new;
      const float alpha = fast_expf_(row.m - m_use);
      p = fast_expf_(s - m_use);
      row.l = row.l * alpha + sw::wave_sum(p);
      row.o[0] *= alpha;
      row.o[1] *= alpha;
      row.m = m_new;
    }
    for (uint64_t left = __ballot(seen); left != 0; left &= left - 1) {            // uniform over the wave
      const int j = __builtin_ctzll(left);
      const float w = __shfl(p, j, 64);
      const uint16_t* v = a.value_cache + (int64_t)__shfl(slot, j, 64) * a.v_stride + (int64_t)g * a.vdim;
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (lane + 64 * b < a.vdim) row.o[b] += w * ld<bf16_t>(v, lane + 64 * b);
    }
  }
  return row;
}

int launch_prompt_attention(const PromptAttention& a, int64_t rows, int max_query_len, hipStream_t stream);

int launch_decode_attention(const PromptAttention& a, int64_t rows, int max_query_len, float* workspace, hipStream_t stream);

}  // namespace swm
