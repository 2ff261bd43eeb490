// KV-cache maintenance kernels for gfx950: reshape_and_cache, copy_blocks,
// swap_blocks, convert_fp8_e5m2.
//
// Semantics follow csrc/cache_kernels.cu of the reference (cited per entry
// point in include/splitwise_hip.h); the tiling does not.  All four are HBM-bound
// byte movers, so the design goal is 16-byte accesses that land in whole 128-byte
// lines:
//   * reshape_and_cache works on tiles of 16 tokens x one head staged through
//     LDS, so that the scatter into the paged layout is issued token-fastest.
//     With consecutive slots (a prompt) one wave store covers contiguous
//     256-byte (K) / 1-KiB (V) pieces of the 4-KiB [block, head] cache tile; with
//     arbitrary slots (decode) every token is still placed individually.
//   * copy_blocks moves 16 bytes per lane with the pointer tables resident on
//     the device (no per-call pointer upload).
#include "common.cuh"

#include <algorithm>
#include <string>
#include <vector>

namespace sw {

namespace {
thread_local std::string g_last_error;
}

void set_error(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
}

constexpr int kTileTokens = 16;
constexpr int kRcThreads = 256;
constexpr size_t kRcLds = 160 * 1024;
// Tokens that the kernel looks at: a tile's, and a vector's behind it.  Its own arrays in LDS: 16 bytes for each, 4 per vector of a tile.
constexpr int rc_group(int vt) { return vt > 0 ? vt : 8; }
constexpr int rc_seen(int vt) { return kTileTokens + rc_group(vt); }
constexpr size_t rc_arrays(int vt) { return (size_t)(16 * rc_seen(vt) + 4 * (kTileTokens / rc_group(vt)) + 15) / 16 * 16; }

// LDS row = head_size activations + 16 bytes of padding (keeps 16-byte row reads
// of consecutive tokens on different bank groups).
template <typename act_t>
__device__ __forceinline__ int lds_row_bytes(int head_size) {
  return head_size * (int)sizeof(typename Conv<act_t>::store_t) + 16;
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
template <typename act_t, bool FP8, int VT>
__global__ void __launch_bounds__(kRcThreads)
reshape_and_cache_tile_kernel(const char* __restrict__ key, const char* __restrict__ value,
                              char* __restrict__ key_cache, char* __restrict__ value_cache,
                              const int64_t* __restrict__ slot_mapping, int num_tokens,
                              int num_heads, int head_size, int block_size, int block_shift,
                              int64_t key_stride_bytes, int64_t value_stride_bytes) {
  using S = typename Conv<act_t>::store_t;
  constexpr int ES = sizeof(S);                 // activation element bytes
  constexpr int CS = FP8 ? 1 : ES;              // cache element bytes
  constexpr int X = 16 / CS;                    // cache elements per 16 bytes
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int GROUP = rc_group(VT), PARTS = kTileTokens / GROUP, kSeen = rc_seen(VT);
  __shared__ int64_t bases[kSeen];              // byte offset of the token's [block, head] tile, -1: no slot
  __shared__ int offsets[kSeen];                // the token's place in its block
  __shared__ int heads[PARTS], loose[kSeen];    // tokens that begin a vector of V, tokens that no vector takes
  static_assert(sizeof(bases) + sizeof(offsets) + sizeof(heads) + sizeof(loose) <= rc_arrays(VT), "the launch counts on them");

  const int t0 = blockIdx.x / num_heads * kTileTokens;
  const int head = blockIdx.x % num_heads;
  const int tid = threadIdx.x;
  const int row_bytes = lds_row_bytes<act_t>(head_size);
  char* k_tile = smem;
  char* v_tile = smem + kTileTokens * row_bytes;
  const int64_t head_bytes = (int64_t)head_size * block_size * CS;
  const int64_t block_bytes = head_bytes * num_heads;

  // ---- every wave looks at the tile's slots, the one in front of them and those up to a vector's length behind: lane l is token
  //      t0 + l - 1
  const int lane = tid & 63, j = lane - 1;
  int64_t slot = -1;
  if (t0 + j >= 0 && t0 + j < num_tokens && j < kSeen) slot = slot_mapping[t0 + j];

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
        uint32_t w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t acc = 0;
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const S e = *reinterpret_cast<const S*>(src + (q * 4 + b) * ES);
            acc |= (uint32_t)Conv<act_t>::to_e5m2(e) << (8 * b);
          }
          w[q] = acc;
        }
        *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
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
      uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < GROUP; ++q) {
        const S e = *reinterpret_cast<const S*>(src + q * row_bytes);
        if constexpr (FP8) {
          w[q >> 2] |= (uint32_t)Conv<act_t>::to_e5m2(e) << (8 * (q & 3));
        } else if constexpr (ES == 2) {
          w[q >> 1] |= (uint32_t)e << (16 * (q & 1));
        } else {
          w[q & 3] = __float_as_uint(e);
        }
      }
      if constexpr (GROUP * CS >= 16) {
        *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
      } else {
        *reinterpret_cast<uint2*>(dst) = make_uint2(w[0], w[1]);
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

// Grid: (2 * num_pairs, num_layers, splits).  blockIdx.x even = K, odd = V.
__global__ void __launch_bounds__(256)
copy_blocks_kernel(const void* const* __restrict__ key_ptrs,
                   const void* const* __restrict__ value_ptrs,
                   const int64_t* __restrict__ mapping, int64_t vecs_per_block) {
  const int pair = blockIdx.x >> 1;
  const bool is_v = blockIdx.x & 1;
  const int layer = blockIdx.y;
  uint4* base = reinterpret_cast<uint4*>(const_cast<void*>(is_v ? value_ptrs[layer] : key_ptrs[layer]));
  const int64_t src = mapping[2 * pair];
  const int64_t dst = mapping[2 * pair + 1];
  const uint4* s = base + src * vecs_per_block;
  uint4* d = base + dst * vecs_per_block;
  for (int64_t i = (int64_t)blockIdx.z * blockDim.x + threadIdx.x; i < vecs_per_block;
       i += (int64_t)gridDim.z * blockDim.x) {
    d[i] = s[i];
  }
}

// 8 elements per lane per step: 16 bytes of f16/bf16 (32 of f32) <-> 8 bytes of e5m2.
template <typename act_t, bool TO_FP8>
__global__ void __launch_bounds__(256)
convert_fp8_e5m2_kernel(const char* __restrict__ src, char* __restrict__ dst, int64_t numel) {
  using S = typename Conv<act_t>::store_t;
  const int64_t nvec = numel / 8;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvec; i += stride) {
    if constexpr (TO_FP8) {
      S e[8];
      if constexpr (sizeof(S) == 2) {
        *reinterpret_cast<uint4*>(e) = reinterpret_cast<const uint4*>(src)[i];
      } else {
        reinterpret_cast<uint4*>(e)[0] = reinterpret_cast<const uint4*>(src)[2 * i];
        reinterpret_cast<uint4*>(e)[1] = reinterpret_cast<const uint4*>(src)[2 * i + 1];
      }
      uint32_t lo = 0, hi = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lo |= (uint32_t)Conv<act_t>::to_e5m2(e[j]) << (8 * j);
        hi |= (uint32_t)Conv<act_t>::to_e5m2(e[4 + j]) << (8 * j);
      }
      reinterpret_cast<uint2*>(dst)[i] = make_uint2(lo, hi);
    } else {
      const uint2 q = reinterpret_cast<const uint2*>(src)[i];
      S e[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        e[j] = Conv<act_t>::from_e5m2((q.x >> (8 * j)) & 0xff);
        e[4 + j] = Conv<act_t>::from_e5m2((q.y >> (8 * j)) & 0xff);
      }
      if constexpr (sizeof(S) == 2) {
        reinterpret_cast<uint4*>(dst)[i] = *reinterpret_cast<uint4*>(e);
      } else {
        reinterpret_cast<uint4*>(dst)[2 * i] = reinterpret_cast<uint4*>(e)[0];
        reinterpret_cast<uint4*>(dst)[2 * i + 1] = reinterpret_cast<uint4*>(e)[1];
      }
    }
  }
  // tail (numel % 8 elements), handled by the first lanes of block 0
  const int64_t tail0 = nvec * 8;
  if (blockIdx.x == 0) {
    for (int64_t i = tail0 + threadIdx.x; i < numel; i += blockDim.x) {
      if constexpr (TO_FP8) {
        reinterpret_cast<uint8_t*>(dst)[i] = Conv<act_t>::to_e5m2(reinterpret_cast<const S*>(src)[i]);
      } else {
        reinterpret_cast<S*>(dst)[i] = Conv<act_t>::from_e5m2(reinterpret_cast<const uint8_t*>(src)[i]);
      }
    }
  }
}

template <typename act_t, bool FP8>
int launch_reshape_and_cache(const void* key, const void* value, void* key_cache, void* value_cache,
                             const int64_t* slot_mapping, int num_tokens, int num_heads,
                             int head_size, int block_size, int64_t key_stride, int64_t value_stride,
                             hipStream_t stream) {
  using S = typename Conv<act_t>::store_t;
  const int es = sizeof(S);
  const int row_bytes = head_size * es + 16;
  const unsigned grid = (unsigned)((num_tokens + kTileTokens - 1) / kTileTokens * num_heads);
  int block_shift = -1;
  if ((block_size & (block_size - 1)) == 0)
    for (block_shift = 0; (1 << block_shift) < block_size; ++block_shift) {}
  // 16 bytes of tokens per store where a block holds a whole number of them, 8 for the small blocks, else single elements
  constexpr int VT = FP8 ? 16 : 16 / (int)sizeof(S);
  int vt = block_size % VT == 0 ? VT : block_size % (VT / 2) == 0 ? VT / 2 : 0;
  // LDS: a tile's rows of K, and of V up to a vector's length less one more (40 rows of 16-bit activations, 48 into an fp8 cache).
  // The largest heads (from 848 on fp32 into fp8, from 2040 on 16 bits) leave room for shorter vectors, or for none.  Without the check
  // a launch that passes 160 KB only with the kernel's own arrays would not be refused but end its queue.
  auto smem = [&](int v) { return (size_t)(2 * kTileTokens + v) * row_bytes; };
  auto fits = [&](int v) { return smem(v) + rc_arrays(v) <= kRcLds; };
  while (vt > 0 && !fits(vt)) vt = vt == VT ? VT / 2 : 0;
  SW_CHECK_ARG(fits(vt), "reshape_and_cache: heads of %d elements need too much LDS", head_size);
  auto kernel = vt == VT  ? reshape_and_cache_tile_kernel<act_t, FP8, VT>
                : vt > 0 ? reshape_and_cache_tile_kernel<act_t, FP8, VT / 2>
                         : reshape_and_cache_tile_kernel<act_t, FP8, 0>;
  kernel<<<grid, kRcThreads, smem(vt), stream>>>(
      static_cast<const char*>(key), static_cast<const char*>(value), static_cast<char*>(key_cache),
      static_cast<char*>(value_cache), slot_mapping, num_tokens, num_heads, head_size, block_size, block_shift,
      key_stride * es, value_stride * es);
  SW_CHECK_LAUNCH();
  return SW_OK;
}

}  // namespace sw

extern "C" {

const char* sw_last_error(void) { return sw::g_last_error.c_str(); }

int sw_abi_version(void) { return 7; }       // SW_ABI_VERSION of the header; tests/test_abi.py compares the two

int sw_get_max_shared_memory_per_block(int device, int* out_bytes) {
  SW_CHECK_ARG(out_bytes != nullptr, "out_bytes is NULL");
  int v = 0;
  SW_CHECK_HIP(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
  *out_bytes = v;
  return SW_OK;
}

int sw_reshape_and_cache(const void* key, const void* value, void* key_cache, void* value_cache,
                         const int64_t* slot_mapping, int num_tokens, int num_heads, int head_size,
                         int block_size, int x, int64_t key_stride, int64_t value_stride,
                         int act_dtype, int cache_dtype, void* stream) {
  using namespace sw;
  if (num_tokens == 0) return SW_OK;
  SW_CHECK_ARG(num_tokens > 0 && num_heads > 0 && head_size > 0 && block_size > 0,
               "reshape_and_cache: bad shape");
  const bool fp8 = cache_dtype == SW_FP8_E5M2;
  SW_CHECK_ARG(act_dtype == SW_F32 || act_dtype == SW_F16 || act_dtype == SW_BF16,
               "Unsupported data type of key/value: %d", act_dtype);
  SW_CHECK_ARG(fp8 || cache_dtype == act_dtype, "Unsupported data type of kv cache: %d", cache_dtype);
  const int es = dtype_size(act_dtype);
  const int cs = fp8 ? 1 : es;
  SW_CHECK_ARG(x == 16 / cs, "reshape_and_cache: x=%d but 16/sizeof(cache element)=%d", x, 16 / cs);
  SW_CHECK_ARG(head_size % x == 0 && (head_size * es) % 16 == 0,
               "reshape_and_cache: head_size %d is not a multiple of x=%d", head_size, x);
  SW_CHECK_ARG((key_stride * es) % 16 == 0 && (value_stride * es) % 16 == 0 &&
                   (reinterpret_cast<uintptr_t>(key) % 16) == 0 &&
                   (reinterpret_cast<uintptr_t>(value) % 16) == 0,
               "reshape_and_cache: key/value rows must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
#define SW_RC(ACT)                                                                              \
  return fp8 ? launch_reshape_and_cache<ACT, true>(key, value, key_cache, value_cache,          \
                                                   slot_mapping, num_tokens, num_heads,         \
                                                   head_size, block_size, key_stride,           \
                                                   value_stride, s)                             \
             : launch_reshape_and_cache<ACT, false>(key, value, key_cache, value_cache,         \
                                                    slot_mapping, num_tokens, num_heads,        \
                                                    head_size, block_size, key_stride,          \
                                                    value_stride, s)
  switch (act_dtype) {
    case SW_F32: SW_RC(float);
    case SW_F16: SW_RC(f16_t);
    default: SW_RC(bf16_t);
  }
#undef SW_RC
}

int sw_copy_blocks(const void* const* key_cache_ptrs, const void* const* value_cache_ptrs,
                   int num_layers, const int64_t* block_mapping, int num_pairs,
                   int64_t block_bytes, void* stream) {
  using namespace sw;
  if (num_layers == 0 || num_pairs == 0) return SW_OK;
  SW_CHECK_ARG(num_layers > 0 && num_pairs > 0 && block_bytes > 0 && block_bytes % 16 == 0,
               "copy_blocks: bad arguments (layers=%d pairs=%d block_bytes=%lld)", num_layers,
               num_pairs, (long long)block_bytes);
  SW_CHECK_ARG(num_layers <= 65535, "copy_blocks: too many layers");
  const int64_t vecs = block_bytes / 16;
  const int splits = (int)std::min<int64_t>(32, std::max<int64_t>(1, vecs / 1024));
  dim3 grid(2 * num_pairs, num_layers, splits);
  copy_blocks_kernel<<<grid, 256, 0, static_cast<hipStream_t>(stream)>>>(
      key_cache_ptrs, value_cache_ptrs, block_mapping, vecs);
  SW_CHECK_LAUNCH();
  return SW_OK;
}

int sw_swap_blocks(const void* src, void* dst, const int64_t* src_blocks, const int64_t* dst_blocks,
                   int n, int64_t block_bytes, int kind, void* stream) {
  using namespace sw;
  if (n == 0) return SW_OK;
  SW_CHECK_ARG(n > 0 && block_bytes > 0, "swap_blocks: bad arguments");
  hipMemcpyKind k;
  switch (kind) {
    case 0: k = hipMemcpyDeviceToDevice; break;
    case 1: k = hipMemcpyDeviceToHost; break;
    case 2: k = hipMemcpyHostToDevice; break;
    default: SW_CHECK_ARG(false, "Invalid device combination");
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  int i = 0;
  while (i < n) {
    int j = i + 1;
    while (j < n && src_blocks[j] == src_blocks[j - 1] + 1 && dst_blocks[j] == dst_blocks[j - 1] + 1) ++j;
    SW_CHECK_HIP(hipMemcpyAsync(static_cast<char*>(dst) + dst_blocks[i] * block_bytes,
                                static_cast<const char*>(src) + src_blocks[i] * block_bytes,
                                (size_t)(j - i) * block_bytes, k, s));
    i = j;
  }
  return SW_OK;
}

int sw_convert_fp8_e5m2(const void* src, void* dst, int64_t numel, int src_dtype, int dst_dtype,
                        void* stream) {
  using namespace sw;
  if (numel == 0) return SW_OK;
  const bool to_fp8 = dst_dtype == SW_FP8_E5M2;
  const int act = to_fp8 ? src_dtype : dst_dtype;
  SW_CHECK_ARG((src_dtype == SW_FP8_E5M2) != (dst_dtype == SW_FP8_E5M2),
               "convert_fp8_e5m2: exactly one side must be fp8_e5m2");
  SW_CHECK_ARG(act == SW_F32 || act == SW_F16 || act == SW_BF16, "convert_fp8_e5m2: bad dtype %d", act);
  SW_CHECK_ARG(reinterpret_cast<uintptr_t>(src) % 16 == 0 && reinterpret_cast<uintptr_t>(dst) % 16 == 0,
               "convert_fp8_e5m2: buffers must be 16-byte aligned");
  const int64_t nvec = std::max<int64_t>(1, numel / 8);
  const int grid = (int)std::min<int64_t>(2048, (nvec + 255) / 256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const char* sp = static_cast<const char*>(src);
  char* dp = static_cast<char*>(dst);
#define SW_CV(ACT)                                                                    \
  if (to_fp8) convert_fp8_e5m2_kernel<ACT, true><<<grid, 256, 0, s>>>(sp, dp, numel); \
  else convert_fp8_e5m2_kernel<ACT, false><<<grid, 256, 0, s>>>(sp, dp, numel);       \
  break
  switch (act) {
    case SW_F32: SW_CV(float);
    case SW_F16: SW_CV(f16_t);
    default: SW_CV(bf16_t);
  }
#undef SW_CV
  SW_CHECK_LAUNCH();
  return SW_OK;
}

}  // extern "C"
