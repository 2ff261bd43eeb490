// Linear attention with one decay per head ("lightning attention"):  S_t = decay_h S_(t-1) + k_t v_t^T,
// o_t = S_t^T q_t, with q, k, v = silu of their projections and the state S [key size, value size] carried in fp32
// per sequence.  A run of new tokens is taken in chunks of 32: inside a chunk the recurrence is three fp32
// matrix products on the matrix cores (v_mfma_f32_32x32x2_f32),
//     A   = (Q K^T) * D,  D[i, j] = decay^(i - j) for j <= i          (tokens of the chunk among themselves)
//     O   = A V + diag(decay^(i + 1)) Q S                              (plus what the carried state holds)
//     S  <- decay^n S + (K * decay^(n - 1 - j))^T V                    (n tokens in the chunk)
// which is the recurrence itself with its sums reordered.  Powers of the decay come from a table built by
// repeated multiplication, never from a quotient, so small decays do not overflow.  The same kernels run "retention":
// the recurrence on fp32 queries and keys that the caller has rotated and scaled, and on the values as they are, no silu.
//
// One wave owns (sequence, head, 32 value channels) and keeps its slice of the state in registers across the
// whole run (the waves of a workgroup share the chunk's queries and keys, staged once in LDS), in the matrix cores' accumulator layout (lane l: value channel l % 32; element r of block b:
// key coordinate 32 b + 8 (r / 4) + 4 (l / 32) + r % 4).  That layout is also what the A operand of S^T q needs
// when q is read in the same order of coordinates, so the state never moves between registers.  Long
// runs are taken by linear_walk.hip (linear_at_most says which), a few tokens by linear_step.hip (linear_step_tokens).
#include "linear_walk.cuh"

#include <climits>

namespace swm {

using f32x16 = __attribute__((ext_vector_type(16))) float;
constexpr int kChunk = 32;

// NDB: 32-coordinate blocks of the key size.  A workgroup owns (sequence, head) and up to 8 blocks of 32 value
// channels, one wave each; the chunk's silu(q) and silu(k) are staged once in LDS for all of them.
// TQ: type of queries and keys (row stride qk_stride), T: of the values (row stride v_stride); SILU: of all three.
template <typename TQ, typename T, bool SILU, int NDB>
__global__ __launch_bounds__(512) void lightning_kernel(
    float* __restrict__ out, const void* __restrict__ q, const void* __restrict__ k, int64_t qk_stride,
    const void* __restrict__ v, int64_t v_stride, const float* __restrict__ decay, float* __restrict__ state, const int32_t* __restrict__ q_start,
    const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ state_slot, int heads, int dim, int vdim, int above, int at_most) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int DS = NDB * 32 + 4;                           // row stride of the staged tiles
  float* Qs = lds;                                           // [32][DS]
  float* Ks = Qs + kChunk * DS;                              // [32][DS]
  float* pw = Ks + kChunk * DS;                              // [kChunk + 1] powers of the decay
  const int h = blockIdx.y;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 31, hl = lane >> 5;
  const int vb = blockIdx.z * (blockDim.x >> 6) + wave;
  // blockIdx.x is a sequence; its whole run goes from the slot's state to the slot's state
  const int seq = blockIdx.x, n = q_start[seq + 1] - q_start[seq];
  if (n <= above || n > at_most) return;                     // the whole workgroup
  const int row0 = q_start[seq];
  const float lam = decay[h];
  if (threadIdx.x == 0) {
    float p = 1.0f;
    for (int e = 0; e <= kChunk; ++e) {
      pw[e] = p;
      p *= lam;
    }
  }
  const int vc = vb * 32 + li;                               // this lane's value channel
  const bool vc_ok = vc < vdim;
  float* sp = state + ((int64_t)state_slot[seq] * heads + h) * (int64_t)dim * vdim;

  f32x16 S[NDB];
  const bool fresh = ctx_len[seq] == 0;
#pragma unroll
  for (int b = 0; b < NDB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int c = 32 * b + 8 * (r / 4) + 4 * hl + (r % 4);
      S[b][r] = (!fresh && vc_ok && c < dim) ? sp[(int64_t)c * vdim + vc] : 0.0f;
    }

  const int64_t qk_col = (int64_t)h * dim, v_col = (int64_t)h * vdim;
  // fp32 operands in pieces of 4
  const bool quads = sizeof(typename Conv<TQ>::store_t) == 4 && dim % 4 == 0 && qk_stride % 4 == 0 &&
                     (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) % 16 == 0;
  for (int c0 = 0; c0 < n; c0 += kChunk) {
    const int cn = min(kChunk, n - c0);
    const int64_t base = (int64_t)(row0 + c0) * qk_stride, v_base = (int64_t)(row0 + c0) * v_stride;
    __syncthreads();                                         // the last chunk's tiles have been read (and pw written)
    if (!SILU && quads) {
      for (int e = threadIdx.x; e < kChunk * NDB * 8; e += blockDim.x) {
        const int r = e / (NDB * 8), c = e % (NDB * 8) * 4;
        float4 qv = make_float4(0.f, 0.f, 0.f, 0.f), kv = qv;
        if (r < cn && c < dim) {
          qv = *reinterpret_cast<const float4*>(static_cast<const float*>(q) + base + r * qk_stride + qk_col + c);
          kv = *reinterpret_cast<const float4*>(static_cast<const float*>(k) + base + r * qk_stride + qk_col + c);
        }
        *reinterpret_cast<float4*>(Qs + r * DS + c) = qv;
        *reinterpret_cast<float4*>(Ks + r * DS + c) = kv;
      }
    } else {
      for (int e = threadIdx.x; e < kChunk * NDB * 32; e += blockDim.x) {
        const int r = e / (NDB * 32), c = e % (NDB * 32);
        float qv = 0.0f, kv = 0.0f;
        if (r < cn && c < dim) {
          qv = ld<TQ>(q, base + r * qk_stride + qk_col + c);
          kv = ld<TQ>(k, base + r * qk_stride + qk_col + c);
          if (SILU) {
            qv = fast_siluf_(qv);
            kv = fast_siluf_(kv);
          }
        }
        Qs[r * DS + c] = qv;
        Ks[r * DS + c] = kv;
      }
    }
    // ---- values of the chunk: channel vc of token (r, hl)
    float vt[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int j = 8 * (r / 4) + 4 * hl + (r % 4);
      const float vv = (vc_ok && j < cn) ? ld<T>(v, v_base + j * v_stride + v_col + vc) : 0.0f;
      vt[r] = SILU ? fast_siluf_(vv) : vv;                   // silu(0) = 0
    }
    __syncthreads();
    // ---- A^T = K Q^T (rows: keys, columns: queries); this lane: token li of the chunk as key and as query
    f32x16 a;
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = 0.0f;
#pragma unroll
    for (int b = 0; b < NDB; ++b) {
      if (32 * b < dim) {
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const int c = 32 * b + 8 * g4 + 4 * hl;
          const float4 qv = *reinterpret_cast<const float4*>(Qs + li * DS + c);
          const float4 kv = *reinterpret_cast<const float4*>(Ks + li * DS + c);
          a = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.x, qv.x, a, 0, 0, 0);
          a = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.y, qv.y, a, 0, 0, 0);
          a = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.z, qv.z, a, 0, 0, 0);
          a = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.w, qv.w, a, 0, 0, 0);
        }
      }
    }
    // element r: key j = 8 (r / 4) + 4 hl + r % 4, query i = li
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int j = 8 * (r / 4) + 4 * hl + (r % 4);
      a[r] = (j <= li && li < cn) ? a[r] * pw[max(li - j, 0)] : 0.0f;
    }
    // ---- O^T = V^T A^T + S^T (Q^T decay^(i + 1))
    f32x16 o;
#pragma unroll
    for (int r = 0; r < 16; ++r) o[r] = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) o = __builtin_amdgcn_mfma_f32_32x32x2f32(vt[r], a[r], o, 0, 0, 0);
    const float carry = pw[li + 1];
#pragma unroll
    for (int b = 0; b < NDB; ++b) {
      if (32 * b < dim) {
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const float4 qv = *reinterpret_cast<const float4*>(Qs + li * DS + 32 * b + 8 * g4 + 4 * hl);
          o = __builtin_amdgcn_mfma_f32_32x32x2f32(S[b][4 * g4], qv.x * carry, o, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_32x32x2f32(S[b][4 * g4 + 1], qv.y * carry, o, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_32x32x2f32(S[b][4 * g4 + 2], qv.z * carry, o, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_32x32x2f32(S[b][4 * g4 + 3], qv.w * carry, o, 0, 0, 0);
        }
      }
    }
    if (li < cn && vb * 32 < vdim) {
      float* dst = out + (int64_t)(row0 + c0 + li) * heads * vdim + v_col + vb * 32;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int c = 8 * (r / 4) + 4 * hl + (r % 4);
        if (vb * 32 + c < vdim) dst[c] = o[r];
      }
    }
    // ---- S <- decay^cn S + (K decay^(cn - 1 - j))^T V : A = keys transposed (coordinate li of block b, token (r, hl))
    const float keep = pw[cn];
#pragma unroll
    for (int b = 0; b < NDB; ++b) {
      if (32 * b < dim) {
#pragma unroll
        for (int r = 0; r < 16; ++r) S[b][r] *= keep;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = 8 * (r / 4) + 4 * hl + (r % 4);
          const float kv = j < cn ? Ks[j * DS + 32 * b + li] * pw[max(cn - 1 - j, 0)] : 0.0f;
          S[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(kv, vt[r], S[b], 0, 0, 0);
        }
      }
    }
  }
  if (vc_ok) {
#pragma unroll
    for (int b = 0; b < NDB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int c = 32 * b + 8 * (r / 4) + 4 * hl + (r % 4);
        if (c < dim) sp[(int64_t)c * vdim + vc] = S[b][r];
      }
  }
}

template <typename TQ, typename T, bool SILU, int NDB>
int launch_lightning(float* out, const void* q, const void* k, int64_t qk_stride, const void* v, int64_t v_stride, const float* decay,
                     float* state, const int32_t* q_start, const int32_t* ctx_len, const int32_t* state_slot,
                     int num_seqs, int heads, int dim, int vdim, int above, int at_most, hipStream_t stream) {
  const int vblocks = (vdim + 31) / 32;
  const int waves = std::min(vblocks, 8);
  const size_t lds_bytes = (size_t)(2 * kChunk * (NDB * 32 + 4) + kChunk + 2) * sizeof(float);
  auto kernel = lightning_kernel<TQ, T, SILU, NDB>;
  static bool raised = false;                                // per instantiation
  if (lds_bytes > 64 * 1024 && !raised) {
    SW_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds_bytes));
    raised = true;
  }
  const unsigned zgroups = (unsigned)((vblocks + waves - 1) / waves);
  hipLaunchKernelGGL(kernel, dim3((unsigned)num_seqs, (unsigned)heads, zgroups), dim3(64 * waves), lds_bytes, stream, out, q, k,
                     qk_stride, v, v_stride, decay, state, q_start, ctx_len, state_slot, heads, dim, vdim, above, at_most);
  SW_CHECK_LAUNCH();
  return SW_OK;
}

}  // namespace swm

extern "C" int64_t swm_lightning_workspace_floats(int64_t rows, int num_seqs, int max_query_len, int heads, int dim,
                                                  int vdim) {
  return swm::linear_walk_plan(false, rows, num_seqs, max_query_len, heads, dim, vdim).floats;
}

extern "C" int swm_lightning(float* out, const void* q, const void* k, const void* v, int64_t in_stride,
                             const float* decay, float* state, const int32_t* q_start, const int32_t* ctx_len,
                             const int32_t* state_slot, int64_t rows, int num_seqs, int max_query_len, int heads,
                             int dim, int vdim, float* workspace, int act_dtype, void* stream) {
  using namespace swm;
  if (rows == 0 || num_seqs == 0) return SW_OK;
  SW_CHECK_ARG(act_ok(act_dtype), "lightning: unsupported dtype %d", act_dtype);
  SW_CHECK_ARG(heads > 0 && heads < 65536 && dim > 0 && dim <= 256 && vdim > 0 && (vdim + 255) / 256 < 65536,
               "lightning: %d heads, key size %d (at most 256), value size %d", heads, dim, vdim);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const LinearWalkPlan plan = linear_walk_plan(false, rows, num_seqs, max_query_len, heads, dim, vdim);
  int at_most = INT_MAX;
  if (workspace != nullptr && plan.at_most < max_query_len) {
    const LinearStep step{out, q, k, v, in_stride, in_stride, state, q_start, ctx_len, state_slot, rows, num_seqs, heads, dim, vdim,
                          workspace};
    const int status = lightning_walk(step, plan, decay, true, act_dtype, act_dtype, s);
    if (status != SW_OK || plan.at_most == 0) return status;
    at_most = plan.at_most;                                  // the others beside it
  }
  int above = 0;                                             // sequences of this many tokens have been seen to
  if (const int few = linear_step_tokens(at_most, rows, num_seqs, max_query_len)) {
    const LinearStep step{out, q, k, v, in_stride, in_stride, state, q_start, ctx_len, state_slot, rows, num_seqs, heads, dim, vdim,
                          nullptr};
    const bool all = few >= std::min(at_most, max_query_len);
    if (lightning_step(step, decay, true, all ? at_most : few, act_dtype, s)) {
      SW_CHECK_LAUNCH();
      if (all) return SW_OK;
      above = few;
    }
  }
#define SWM_LIGHTNING_CASE(N)                                                                                              \
  case N:                                                                                                                  \
    SWM_DISPATCH_ACT(act_dtype, return (launch_lightning<T, T, true, N>(out, q, k, in_stride, v, in_stride, decay, state,  \
                                                                        q_start, ctx_len, state_slot, num_seqs, heads,     \
                                                                        dim, vdim, above, at_most, s)););                         \
    break;
  switch ((dim + 31) / 32) {
    SWM_LIGHTNING_CASE(1)
    SWM_LIGHTNING_CASE(2)
    SWM_LIGHTNING_CASE(3)
    SWM_LIGHTNING_CASE(4)
    SWM_LIGHTNING_CASE(5)
    SWM_LIGHTNING_CASE(6)
    SWM_LIGHTNING_CASE(7)
    SWM_LIGHTNING_CASE(8)
  }
#undef SWM_LIGHTNING_CASE
  return SW_OK;
}

extern "C" int swm_retention(float* out, const float* q, const float* k, int64_t qk_stride, const void* v, int64_t v_stride,
                             const float* decay, float* state, const int32_t* q_start, const int32_t* ctx_len,
                             const int32_t* state_slot, int64_t rows, int num_seqs, int max_query_len, int heads, int dim,
                             int vdim, float* workspace, int act_dtype, void* stream) {
  using namespace swm;
  if (rows == 0 || num_seqs == 0) return SW_OK;
  SW_CHECK_ARG(act_ok(act_dtype), "retention: unsupported dtype %d", act_dtype);
  SW_CHECK_ARG(heads > 0 && heads < 65536 && dim > 0 && dim <= 256 && vdim > 0 && (vdim + 255) / 256 < 65536,
               "retention: %d heads, key size %d (at most 256), value size %d", heads, dim, vdim);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const LinearWalkPlan plan = linear_walk_plan(false, rows, num_seqs, max_query_len, heads, dim, vdim);
  int at_most = INT_MAX;
  if (workspace != nullptr && plan.at_most < max_query_len) {
    const LinearStep step{out, q, k, v, qk_stride, v_stride, state, q_start, ctx_len, state_slot, rows, num_seqs, heads, dim, vdim,
                          workspace};
    const int status = lightning_walk(step, plan, decay, false, SW_F32, act_dtype, s);
    if (status != SW_OK || plan.at_most == 0) return status;
    at_most = plan.at_most;                                  // the others beside it
  }
  int above = 0;                                             // sequences of this many tokens have been seen to
  if (const int few = linear_step_tokens(at_most, rows, num_seqs, max_query_len)) {
    const LinearStep step{out, q, k, v, qk_stride, v_stride, state, q_start, ctx_len, state_slot, rows, num_seqs, heads, dim, vdim,
                          nullptr};
    const bool all = few >= std::min(at_most, max_query_len);
    if (lightning_step(step, decay, false, all ? at_most : few, act_dtype, s)) {
      SW_CHECK_LAUNCH();
      if (all) return SW_OK;
      above = few;
    }
  }
#define SWM_RETENTION_CASE(N)                                                                                          \
  case N:                                                                                                              \
    SWM_DISPATCH_ACT(act_dtype, return (launch_lightning<float, T, false, N>(out, q, k, qk_stride, v, v_stride, decay, \
                                                                             state, q_start, ctx_len, state_slot,      \
                                                                             num_seqs, heads, dim, vdim, above, at_most, s)););\
    break;
  switch ((dim + 31) / 32) {
    SWM_RETENTION_CASE(1)
    SWM_RETENTION_CASE(2)
    SWM_RETENTION_CASE(3)
    SWM_RETENTION_CASE(4)
    SWM_RETENTION_CASE(5)
    SWM_RETENTION_CASE(6)
    SWM_RETENTION_CASE(7)
    SWM_RETENTION_CASE(8)
  }
#undef SWM_RETENTION_CASE
  return SW_OK;
}
