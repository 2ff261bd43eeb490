// A tile of the cache write: 16 tokens of a run of neighbouring heads into the paged layout, by 256 threads.  Used by reshape_and_cache
// (cache_kernels.hip) and by prompt attention, which writes the cache beside its own work (prefill_attention.hip).
#pragma once

#include "common.cuh"

namespace sw {

constexpr int kTileTokens = 16;
constexpr int kRcThreads = 256;
constexpr size_t kRcLds = 160 * 1024;
// Tokens that a tile looks at: its own, and a vector's behind it.  Its arrays in LDS: 16 bytes for each, 4 per vector of a tile.
__host__ __device__ constexpr int rc_group(int vt) { return vt > 0 ? vt : 8; }
__host__ __device__ constexpr int rc_seen(int vt) { return kTileTokens + rc_group(vt); }
__host__ __device__ constexpr size_t rc_arrays(int vt) { return (size_t)(16 * rc_seen(vt) + 4 * (kTileTokens / rc_group(vt)) + 15) / 16 * 16; }
// ... and its rows of K, and of V up to a vector's length less one more (40 rows of 16-bit activations, 48 into an fp8 cache), each with
// 16 bytes of padding (16-byte reads of consecutive tokens' rows are on different bank groups)
__host__ __device__ constexpr size_t rc_lds(int vt, int row_elements, int element_bytes) {
  return rc_arrays(vt) + (size_t)(2 * kTileTokens + vt) * (row_elements * element_bytes + 16);
}

// Heads that lie side by side in a token's row do so in a block of the cache too: `num_heads` heads of `head_size` are as well half as
// many of twice the size.  Beside the attention a tile takes as many of them as a row of 1 KB holds and as leave a launch enough tiles
// (cache_merge); alone it takes one, of which more fit on a compute unit.
struct CacheWrite {
  const char *key, *value;
  char *key_cache, *value_cache;
  const int64_t* slot_mapping;
  int num_tokens, num_heads, head_size, block_size, block_shift;
  int64_t key_stride_bytes, value_stride_bytes;
  int tiles() const { return (num_tokens + kTileTokens - 1) / kTileTokens * num_heads; }
};
inline CacheWrite cache_write(const void* key, const void* value, void* key_cache, void* value_cache, const int64_t* slot_mapping,
                              int num_tokens, int num_heads, int head_size, int block_size, int64_t key_stride, int64_t value_stride,
                              int element_bytes) {
  CacheWrite w{static_cast<const char*>(key), static_cast<const char*>(value), static_cast<char*>(key_cache),
               static_cast<char*>(value_cache), slot_mapping, num_tokens, num_heads, head_size, block_size, -1,
               key_stride * element_bytes, value_stride * element_bytes};
  if ((block_size & (block_size - 1)) == 0)
    for (w.block_shift = 0; (1 << w.block_shift) < block_size; ++w.block_shift) {}
  return w;
}
// at_least: tiles that are to be left; lds: bytes that a tile may have
inline void cache_merge(CacheWrite& w, int vt, int element_bytes, int at_least, size_t lds) {
  while (w.num_heads % 2 == 0 && 2 * w.head_size * element_bytes <= 1024 && w.tiles() / 2 >= at_least &&
         rc_lds(vt, 2 * w.head_size, element_bytes) <= lds) {
    w.num_heads /= 2;
    w.head_size *= 2;
  }
}

// act_t: float / f16_t / bf16_t.  FP8: cache holds e5m2 bytes, else the same bits as the activations.  VT: tokens per vector
// store of a value cache row (0: element by element).
// What bounds it is memory, once the addresses are cheap: where a token goes (its slot's block and offset, a 64-bit division
// where the block size is no power of two) is worked out once per tile by 16 lanes, and not by every thread for every piece.
// Workgroups that run together take the heads of the same tokens: their pieces of a row lie side by side.
// Vectors of V are VT neighbouring slots from a multiple of VT on.  Prompts of any length lie behind one another in a step, so a
// tile's tokens seldom begin at such a slot: a tile's V is moved on to the next one where the run of slots goes on (its first
// tokens are then the tile's before it), and only what is left over at a run's ends goes element by element.
// Measured, 2320 tokens x 32 heads of 128, bf16 (76 MB): 30.5 us with the divisions in every thread, 27.2 without, 16.2 with the
// heads side by side as one prompt; as prompts of 699, 938 and 790 tokens 26.0 with V vectors only where a tile's own eighths
// are aligned, 18.3 here.  61 tokens x 8 heads into an fp8 cache: 8.7 us with the divisions, 5.1 here.  251 tokens x 32 heads into slots of their own
// take 19 us before and after: every element of V is a 2-byte write into a 32-byte sector (36 MB for 4).
// tid: 0 .. 255; smem: rc_lds bytes on 16 bytes.  All threads of the workgroup meet in here, a tile behind the last one has no tokens.
template <typename act_t, bool FP8, int VT>
__device__ __forceinline__ void cache_tile(const CacheWrite& w, int tile, int tid, char* smem) {
  const char *const key = w.key, *const value = w.value;
  char *const key_cache = w.key_cache, *const value_cache = w.value_cache;
  const int num_tokens = w.num_tokens, num_heads = w.num_heads, head_size = w.head_size, block_size = w.block_size,
            block_shift = w.block_shift;
  const int64_t key_stride_bytes = w.key_stride_bytes, value_stride_bytes = w.value_stride_bytes;
  using S = typename Conv<act_t>::store_t;
  constexpr int ES = sizeof(S);                 // activation element bytes
  constexpr int CS = FP8 ? 1 : ES;              // cache element bytes
  constexpr int X = 16 / CS;                    // cache elements per 16 bytes
  constexpr int GROUP = rc_group(VT), PARTS = kTileTokens / GROUP, kSeen = rc_seen(VT);
  int64_t* const bases = reinterpret_cast<int64_t*>(smem);   // [kSeen] byte offset of the token's [block, head] tile, -1: no slot
  int* const offsets = reinterpret_cast<int*>(bases + kSeen);            // [kSeen] the token's place in its block
  int* const loose = offsets + kSeen;           // [kSeen] tokens that no vector of V takes
  int* const heads = loose + kSeen;             // [PARTS] tokens that begin one

  const int t0 = tile / num_heads * kTileTokens;
  const int head = tile % num_heads;
  const int row_bytes = head_size * ES + 16;
  char* k_tile = smem + rc_arrays(VT);
  char* v_tile = k_tile + kTileTokens * row_bytes;
  const int64_t head_bytes = (int64_t)head_size * block_size * CS;
  const int64_t block_bytes = head_bytes * num_heads;

  // ---- every wave looks at the tile's slots, the one in front of them and those up to a vector's length behind: lane l is token
  //      t0 + l - 1
  const int lane = tid & 63, j = lane - 1;
  int64_t slot = -1;
  if (t0 + j >= 0 && t0 + j < num_tokens && j < kSeen) slot = w.slot_mapping[t0 + j];

  // ---- stage K and V rows of this head: 16-byte pieces, token-major (coalesced), 16 lanes a row
  const int tok16 = tid / 16, chunks = head_size * ES / 16;
  const int64_t head_off = (int64_t)head * head_size * ES;
  if (t0 + tok16 < num_tokens) {
    const char* kr = key + (t0 + tok16) * key_stride_bytes + head_off;
    const char* vr = value + (t0 + tok16) * value_stride_bytes + head_off;
    for (int ch = tid % 16; ch < chunks; ch += 16) {
      const uint4 kv = *reinterpret_cast<const uint4*>(kr + ch * 16);
      const uint4 vv = *reinterpret_cast<const uint4*>(vr + ch * 16);
      *reinterpret_cast<uint4*>(k_tile + tok16 * row_bytes + ch * 16) = kv;
      *reinterpret_cast<uint4*>(v_tile + tok16 * row_bytes + ch * 16) = vv;
    }
  }
  // ---- V's tokens [v0, v1) of this tile, which of them begin a vector and which go alone
  const int64_t prev = __shfl_up(slot, 1, 64);
  const uint64_t follows = __ballot(lane > 0 && slot >= 0 && prev >= 0 && slot == prev + 1);
  auto moved = [&](int first) {                 // tokens from `first` on that belong to a vector begun in front of it
    if constexpr (VT == 0) return 0;
    const int64_t s = __shfl(slot, first + 1, 64);
    const int n = s < 0 ? 0 : (int)((GROUP - s % GROUP) % GROUP);
    const uint64_t need = ((1ull << n) - 1) << (first + 1);
    return (follows & need) == need ? n : 0;
  };
  const int v0 = moved(0), v1 = min(kTileTokens + moved(kTileTokens), num_tokens - t0);
  uint64_t begins = 0;
  if constexpr (VT > 0) {
    const uint64_t rest = ((1ull << (GROUP - 1)) - 1) << (lane + 1);
    begins = __ballot(j >= v0 && j + GROUP <= v1 && slot >= 0 && slot % GROUP == 0 && (follows & rest) == rest);
  }
  const bool taken = ((begins << (GROUP - 1)) >> lane & ((1ull << GROUP) - 1)) != 0;
  const uint64_t alone = __ballot(j >= v0 && j < v1 && slot >= 0 && !taken);
  const int num_heads_v = __popcll(begins), num_loose = __popcll(alone);
  if (tid < 64) {                               // one wave
    const uint64_t below = (1ull << lane) - 1;
    if (begins >> lane & 1) heads[__popcll(begins & below)] = j;
    if (alone >> lane & 1) loose[__popcll(alone & below)] = j;
    if (j >= 0 && j < kSeen) {
      const int64_t blk = block_shift >= 0 ? slot >> block_shift : slot / block_size;
      bases[j] = slot < 0 ? -1 : blk * block_bytes + head * head_bytes;
      offsets[j] = slot < 0 ? 0 : (int)(slot - blk * block_size);
    }
  }
  if (kTileTokens + tok16 < v1) {               // (fewer than a vector's tokens)
    const char* vr = value + (t0 + kTileTokens + tok16) * value_stride_bytes + head_off;
    for (int ch = tid % 16; ch < chunks; ch += 16)
      *reinterpret_cast<uint4*>(v_tile + (kTileTokens + tok16) * row_bytes + ch * 16) = *reinterpret_cast<const uint4*>(vr + ch * 16);
  }
  __syncthreads();

  // ---- K: one 16-byte cache vector (X elements of one token) per lane, token-fastest
  {
    const int tok = tid % kTileTokens;
    const int64_t base = bases[tok];
    const int boff = offsets[tok];
    for (int c = tid / kTileTokens; base >= 0 && c < head_size / X; c += kRcThreads / kTileTokens) {
      char* dst = key_cache + base + ((int64_t)c * block_size + boff) * 16;
      const char* src = k_tile + tok * row_bytes + c * X * ES;
      if constexpr (!FP8) {
        *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
      } else {
        uint32_t words[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t acc = 0;
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const S e = *reinterpret_cast<const S*>(src + (q * 4 + b) * ES);
            acc |= (uint32_t)Conv<act_t>::to_e5m2(e) << (8 * b);
          }
          words[q] = acc;
        }
        *reinterpret_cast<uint4*>(dst) = make_uint4(words[0], words[1], words[2], words[3]);
      }
    }
  }

  // ---- V: cache row d holds block_size tokens.  A vector takes VT tokens of it (block_size is a multiple: they share a row segment),
  // what no vector takes goes one element per lane.
  const int part = tid % PARTS;
  if (part < num_heads_v) {
    const int first = heads[part];
    char* const dst0 = value_cache + bases[first] + (int64_t)offsets[first] * CS;
    for (int d = tid / PARTS; d < head_size; d += kRcThreads / PARTS) {
      const char* src = v_tile + first * row_bytes + d * ES;
      char* dst = dst0 + (int64_t)d * block_size * CS;
      uint32_t words[4] = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < GROUP; ++q) {
        const S e = *reinterpret_cast<const S*>(src + q * row_bytes);
        if constexpr (FP8) {
          words[q >> 2] |= (uint32_t)Conv<act_t>::to_e5m2(e) << (8 * (q & 3));
        } else if constexpr (ES == 2) {
          words[q >> 1] |= (uint32_t)e << (16 * (q & 1));
        } else {
          words[q & 3] = __float_as_uint(e);
        }
      }
      if constexpr (GROUP * CS >= 16) {
        *reinterpret_cast<uint4*>(dst) = make_uint4(words[0], words[1], words[2], words[3]);
      } else {
        *reinterpret_cast<uint2*>(dst) = make_uint2(words[0], words[1]);
      }
    }
  }
#pragma unroll 4
  for (int k = tid / 64; k < num_loose; k += kRcThreads / 64) {          // a wave per token
    const int tok = __builtin_amdgcn_readfirstlane(loose[k]);
    char* const dst0 = value_cache + bases[tok] + (int64_t)offsets[tok] * CS;
    for (int d = lane; d < head_size; d += 64) {
      char* dst = dst0 + (int64_t)d * block_size * CS;
      const S e = *reinterpret_cast<const S*>(v_tile + tok * row_bytes + d * ES);
      if constexpr (FP8) {
        *reinterpret_cast<uint8_t*>(dst) = Conv<act_t>::to_e5m2(e);
      } else {
        *reinterpret_cast<S*>(dst) = e;
      }
    }
  }
}

}  // namespace sw
