// Which kernels a step of the paged attention goes to (capped_attention.hip).  Host code, no HIP headers.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace swm {

constexpr int kAttentionTile = 32;      // query rows of a tile
constexpr int kPromptWaves = 4;         // tiles of a workgroup of the prompt kernel
// Decode steps on the matrix cores: at most this many query rows (tokens x heads of a group) per sequence and key/value head
constexpr int kDecodeRows = 8;
constexpr int kDecodeGroups = 256, kDecodePartKeys = 256, kDecodeSharedKeys = 1024;

enum AttentionWay {
  kPromptOnMatrixCores,                 // prompt_attention.hip
  kDecodeOnMatrixCores,                 // decode_attention.hip
  kGeneralAttention                     // capped_attention.hip
};

// an upper bound of the keys that a query sees
inline int64_t attention_most_keys(int max_query_len, int page_size, int table_width, int window, int chunk) {
  int64_t most = (int64_t)page_size * table_width;
  if (window > 0) most = std::min<int64_t>(most, window + max_query_len);
  if (chunk > 0) most = std::min<int64_t>(most, chunk);
  return most;
}

// Whether the bf16 matrix kernels can take a step: a bf16 cache whose rows can be read in 16-byte pieces, key and value sizes up
// to 128.  Beyond 128 the three parts of a prompt's queries (96 registers at 128) no longer leave room for two waves per SIMD;
// fp32 caches have no exact bf16 keys.  Both keep the general kernels.  addresses: those of queries, keys and values, or'ed.
inline bool attention_pieces(uintptr_t addresses, int dim, int vdim, int64_t k_stride, int64_t v_stride) {
  return dim <= 128 && vdim <= 128 && dim % 8 == 0 && vdim % 8 == 0 && k_stride % 8 == 0 && v_stride % 8 == 0 && addresses % 16 == 0;
}

// Steps of one query row per sequence and key/value head over few keys: the vector kernel has no parts to make, nothing to lay side
// by side and less to join.  Up to how many keys, measured (us a step, vector / matrix; one sequence and 250, 8 heads each):
//   128 wide:  16 keys 7.0 / 7.9 and 40 / 54, 256 keys 9.2 / 10.7 and 80 / 89, 511 keys 11.8 / 12.8 and 140 / 144, 801 keys 15.8 /
//              15.2 and 198 / 186
//   64 wide:   128 keys 6.0 / 6.4 and 25.1 / 27.7, 256 keys 6.8 / 7.0 and 31.9 / 35.2, 511 keys 8.7 / 8.3 and 50.5 / 48.1
//   32 wide:   64 keys 4.9 / 5.0 and 15.1 / 18.4, 128 keys 5.4 / 5.1 and 18.0 / 20.7, 144 keys of one 5.2 / 5.5, 301 keys 6.6 / 6.0
//              and 32.4 / 33.1
//   96 wide (a block of 32 fewer for the matrix cores, but not for the vector kernel's lanes):  64 keys 7.4 / 7.4 and 46 / 51, 143
//              keys 8.0 / 8.2 and 57 / 63, 256 keys 8.9 / 9.1 and 76 / 76
// With more rows (two and more heads a group) the matrix cores win at once: 4 sequences, 8 heads on 4 of 64, 17 keys 7.2 / 6.1.
// groups: sequences x heads.  The matrix kernel has two workgroups, of a group each, on a compute unit, 512 at once; up to 64 wide a
// few more groups than that make a second round of it, nearly empty: 12 heads of 64, 60 sequences, 16 keys 7.5 / 10.1, 301 keys 16.8 /
// 18.1, 801 keys 28.7 / 28.7;  10 heads of 64, 55 sequences, 1001 keys 28.5 / 31.3.
inline int attention_one_row_keys(int64_t groups, int dim, int vdim) {
  const int size = std::max(dim, vdim);
  if (size > 64) return size > 96 ? 512 : 160;
  if (groups > 512 && groups <= 768) return 1024;
  return groups > 1024 ? 320 : size > 32 ? 256 : 160;
}

// The larger of a page's bytes of keys and of values (bf16), from one slot to the next of the same place.
inline int64_t attention_page_bytes(int page_size, int64_t k_stride, int64_t v_stride) {
  return 2 * (int64_t)page_size * std::max(k_stride, v_stride);
}

// max_query_len 0: unknown.  pieces: attention_pieces of a bf16 cache.  page_bytes: the prompt kernel has a key's place in its page in
// 32 bits (64-bit products took a seventh of its vector units' time); a page of 4 GiB and more goes to the general kernel.
inline AttentionWay attention_way(bool pieces, int num_seqs, int max_query_len, int heads, int kv_heads, int dim, int vdim,
                                  int page_size, int table_width, int window, int chunk, int64_t page_bytes = 0) {
  const int group = heads / kv_heads;
  if (!pieces) return kGeneralAttention;
  if (max_query_len <= 0 || max_query_len > kAttentionTile / group)
    return page_bytes < (int64_t)1 << 32 ? kPromptOnMatrixCores : kGeneralAttention;
  if (max_query_len * group > kDecodeRows) return kGeneralAttention;
  if (max_query_len * group == 1 && attention_most_keys(max_query_len, page_size, table_width, window, chunk) <=
                                        attention_one_row_keys((int64_t)num_seqs * kv_heads, dim, vdim))
    return kGeneralAttention;
  return kDecodeOnMatrixCores;
}

// The prompt kernel's workgroups, an upper bound: tiles of every sequence's tokens for every key/value head.
inline int prompt_tokens(int heads, int kv_heads) { return kPromptWaves * (kAttentionTile / (heads / kv_heads)); }
inline int64_t prompt_attention_workgroups(int64_t rows, int num_seqs, int heads, int kv_heads) {
  const int tokens = prompt_tokens(heads, kv_heads);
  return ((rows + tokens - 1) / tokens + num_seqs) * kv_heads;
}

// How many groups of waves share a workgroup's walk in the prompt kernel, 1 or 2.  Two shorten the longest walk, which is what a launch
// waits for that leaves it a compute unit of its own; but only one such workgroup fits a compute unit, where of one group's two do, and
// those fill one another's gaps better than two groups do (by 5 to 12 % where a launch has many rounds of them).
// Measured in 1435 steps (us, one group / two; W: workgroups, as counted above; 16 query heads on 4 of 128 unless stated):
//   Keys, an upper bound of the longest walk (the block tables' width, the mask): below 256 the two cost more than they save (80 steps,
//   0.96 on average): one prompt of 77 tokens, 8 heads on 2: 18.2 / 20.3; from there on they gain, 271 twice, 12 on 4 of 64: 20.3 / 18.4.
//   W up to 256, a compute unit for each: 1.19 on average whatever the mask, the lengths and the decoding sequences beside: 64 tokens
//   behind 1406, window 256 25.4 / 23.7, 1766 tokens 110.7 / 92.2, 723 tokens six times, 8 on 2, window 256 (W 238) 26.8 / 27.3; about a
//   hundred decoding sequences over 500 keys each lose up to 5 % (W 135, 8 on 1 of 64, 35.9 / 37.8).
//   Beyond, a second round begins where the first one's short walks end: the causal mask's, of tiles at the front of a sequence.  That
//   pays where the longest sequence has at least half of the workgroups and there are few of one token: 3446 tokens (W 436) 201.8 /
//   154.1, 1419 and 1903 (W 424) 129.5 / 94.9; not with 950 at most of five sequences (W 464) 63.8 / 73.4, with ten decoding sequences
//   beside 3520 tokens (W 488) 202 / 258, 371 tokens six times, 32 on 8 (W 512), 35.1 / 46.1, and not
//   under a window or chunks of fewer keys (20 steps, 0.75 to 1.26).
//   With keys in front of the prompt walks are less uneven: up to W 512 1.01 to 1.33, beyond 0.84 to 1.05 (2271 behind 1047, 32 on 8,
//   W 576: 242 / 288).  Without, 1.25 to 1.33 on average up to W 512, 1.12 (1.01 to 1.30) from 544 to 560, 1.08 (0.94 to 1.23) to 576,
//   1.01 (0.86 to 1.14) from 592 to 608, 0.98 from 640 on.
constexpr int64_t kSharedWalkKeys = 256, kSharedWalksAlone = 256, kSharedWalksBehind = 512, kSharedWalks = 560;
inline int prompt_attention_groups(int64_t rows, int num_seqs, int max_query_len, int heads, int kv_heads, int page_size, int table_width,
                                   int window, int chunk) {
  const int64_t keys = (int64_t)table_width * page_size, mask = window > 0 ? window : chunk > 0 ? chunk : keys;
  const int64_t all = prompt_attention_workgroups(rows, num_seqs, heads, kv_heads);
  if (std::min(keys, mask) < kSharedWalkKeys) return 1;
  if (all <= kSharedWalksAlone) return 2;
  const int tokens = prompt_tokens(heads, kv_heads);
  const int64_t longest = (int64_t)((max_query_len + tokens - 1) / tokens) * kv_heads;
  const bool whole = keys - page_size <= (int64_t)max_query_len * 5 / 4;       // next to nothing in front of the longest prompt
  return mask >= keys && 2 * longest >= all && 16 * (int64_t)num_seqs * kv_heads <= all && all <= (whole ? kSharedWalks : kSharedWalksBehind)
             ? 2 : 1;
}

// How many workgroups share a sequence's keys in the decode kernel on the matrix cores, given a workspace of parts x rows x heads x
// (vdim + 2) floats.
// One workgroup per compute unit and no more: its waves have 128 KB under way.  Two for each made 61 sequences of 2041 keys, 16
// heads on 4, 67 us instead of 61 and 9 sequences on 8 key/value heads 28 instead of 23 (the join, and shorter runs).  A part has at
// least a tile a wave.  Below about 1024 keys the second launch costs more than the sharing saves: 2 sequences of 700 keys 20.3 us
// shared and 16.0 alone, 3 of 1000 20.5 and 21.2, 2 of 2500 20.5 and 22.7 (shared among a fourth as many).
inline int decode_attention_parts(int num_seqs, int max_query_len, int heads, int kv_heads, int page_size, int table_width,
                                  int window, int chunk) {
  if (max_query_len <= 0 || (int64_t)max_query_len * (heads / kv_heads) > kDecodeRows) return 1;
  const int64_t most_keys = attention_most_keys(max_query_len, page_size, table_width, window, chunk);
  if (most_keys < kDecodeSharedKeys) return 1;
  const int64_t groups = (int64_t)num_seqs * kv_heads;
  int parts = 1;
  while (parts < 16 && groups * parts * 2 <= kDecodeGroups && most_keys >= 2 * parts * kDecodePartKeys) parts <<= 1;
  return parts;
}

}  // namespace swm
