// Steps of capped_attention.hip that run on the bf16 matrix cores, prompts (prompt_attention.hip) and decode steps of few rows
// (decode_attention.hip): arguments and dispatch.
#pragma once

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

// Whether a step goes there: a bf16 cache whose rows can be read in 16-byte pieces, key and value sizes up to 128.  Beyond 128
// the three parts of a prompt's queries (96 registers at 128) no longer leave room for two waves per SIMD; fp32 caches have no
// exact bf16 keys.  Both keep the general kernels.
inline bool prompt_attention_fits(const float* q, const void* key_cache, const void* value_cache, int dim, int vdim,
                                  int64_t k_stride, int64_t v_stride) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(key_cache) |
                       reinterpret_cast<uintptr_t>(value_cache);
  return dim <= 128 && vdim <= 128 && dim % 8 == 0 && vdim % 8 == 0 && k_stride % 8 == 0 && v_stride % 8 == 0 && at % 16 == 0;
}

int launch_prompt_attention(const PromptAttention& a, int64_t rows, hipStream_t stream);

// Decode steps: at most this many query rows (tokens x heads of a group) per sequence and key/value head
constexpr int kDecodeRows = 8;
constexpr int kDecodeGroups = 256, kDecodePartKeys = 256, kDecodeSharedKeys = 1024;
// how many workgroups share a sequence's keys, given a workspace of parts x rows x heads x (vdim + 2) floats
int decode_attention_parts(int num_seqs, int max_query_len, int heads, int kv_heads, int page_size, int table_width, int window,
                           int chunk);
int launch_decode_attention(const PromptAttention& a, int64_t rows, int max_query_len, float* workspace, hipStream_t stream);

}  // namespace swm
