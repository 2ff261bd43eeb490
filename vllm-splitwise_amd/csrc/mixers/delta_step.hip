// One decode step of the delta rule with decays (one per head, or one per key channel), prologue included:
//     S <- diag(g) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q            (S [dim, vdim] fp32, q, k made unit vectors)
// What bounds it: the states, which are read and written once.  A workgroup owns (sequence, head) and CW neighbouring value
// channels; thread (group, piece) holds the rows group, group + G, ... of 4 neighbouring channels in registers, so a wave reads
// and writes the state in whole rows of 16-byte pieces, every load in flight before the first is used.  The key products
// meet in LDS across the groups.  q, k and the decays are worked out by the workgroup itself while the state is on its way:
// the launch of a prologue and its operands' trip through memory go.
// Measured, 61 sequences x 16 heads of 128 x 128 (128 MB of states read and written), convolution, norm and gate included: 100 us
// as a prologue and a recurrence with 16 columns per wave read in pieces of 64 bytes (1.3 TB/s), 39 us here.
// Longer runs of tokens are walked token by token with the state staying in registers.
#include "delta_step.h"
#include "mixers_common.cuh"

#include <algorithm>

namespace swm {

constexpr int kStepThreads = 256;

// R: rows per thread (dim <= R * groups)
template <typename T, int R>
__global__ __launch_bounds__(kStepThreads) void delta_step_kernel(
    float* __restrict__ out, const float* __restrict__ qkv, const void* __restrict__ beta_pre, int64_t beta_stride,
    const void* __restrict__ decay_pre, int64_t decay_stride, int decay_per_head, const float* __restrict__ dt_bias,
    const float* __restrict__ a_log, float* __restrict__ state, const int32_t* __restrict__ q_start,
    const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ state_slot, int heads, int kv_heads, int dim, int vdim,
    int lanes, int at_most) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int groups = kStepThreads / lanes;                   // lanes: threads across the value channels, a power of two
  float* Q = lds;                                            // [dim] unit query times dim^-1/2
  float* K = Q + dim;                                        // [dim] unit key
  float* D = K + dim;                                        // [dim] decays
  float* part = lds + (3 * dim + 3) / 4 * 4;                 // [groups][lanes * 4]
  float* red = part + kStepThreads * 4;                      // [4][2]
  const int h = blockIdx.y, s = blockIdx.z;
  const int first = q_start[s], n = q_start[s + 1] - first;
  if (n <= 0 || n > at_most) return;                         // the whole workgroup
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int piece = tid % lanes, group = tid / lanes;
  const int col = (blockIdx.x * lanes + piece) * 4;
  const bool col_ok = col < vdim;                            // vdim is a multiple of 4
  float* S = state + ((int64_t)state_slot[s] * heads + h) * (int64_t)dim * vdim;           // uniform; 32-bit offsets from it
  const uint32_t at0 = (uint32_t)(group * vdim + col), hop = (uint32_t)(groups * vdim);
  const bool carried = ctx_len[s] > 0;
  float4 x[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = group + i * groups;
    x[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (carried && col_ok && row < dim) x[i] = *reinterpret_cast<const float4*>(S + (at0 + i * hop));
  }
  const int64_t row_w = 2 * (int64_t)kv_heads * dim + (int64_t)heads * vdim;
  const int c = h / (heads / kv_heads);
  const float rate = expf(a_log[h]), qscale = 1.0f / sqrtf((float)dim);
  for (int t = 0; t < n; ++t) {
    const int64_t tok = first + t;
    const float* q = qkv + tok * row_w + (int64_t)c * dim;
    const float* k = q + (int64_t)kv_heads * dim;
    // ---- unit query and key, decays; every thread ends up with beta and the sums
    const float qv = tid < dim ? q[tid] : 0.0f, kv = tid < dim ? k[tid] : 0.0f;          // dim <= 256
    const float qq = sw::wave_sum(qv * qv), kk = sw::wave_sum(kv * kv);
    const float4 v = col_ok ? *reinterpret_cast<const float4*>(qkv + tok * row_w + 2 * (int64_t)kv_heads * dim + (int64_t)h * vdim + col)
                            : make_float4(0.f, 0.f, 0.f, 0.f);
    const float beta = sigmoidf_(ld<T>(beta_pre, tok * beta_stride + h));
    float g = 0.0f;
    if (tid < dim) {
      const int at = decay_per_head ? h : h * dim + tid;
      g = expf(-rate * softplusf_(ld<T>(decay_pre, tok * decay_stride + at) + dt_bias[at]));
    }
    __syncthreads();                                         // the last token's sums have been read
    if (lane == 0) {
      red[wave * 2] = qq;
      red[wave * 2 + 1] = kk;
    }
    __syncthreads();
    float sq = 0.0f, sk = 0.0f;
#pragma unroll
    for (int w = 0; w < kStepThreads / 64; ++w) {
      sq += red[2 * w];
      sk += red[2 * w + 1];
    }
    if (tid < dim) {
      Q[tid] = qv * (qscale / sqrtf(sq + 1e-6f));
      K[tid] = kv * (1.0f / sqrtf(sk + 1e-6f));
      D[tid] = g;
    }
    __syncthreads();
    // ---- S <- diag(g) S, its product with the key
    float4 ks = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int row = group + i * groups;
      if (row < dim) {
        const float gr = D[row], kr = K[row];
        x[i].x *= gr; x[i].y *= gr; x[i].z *= gr; x[i].w *= gr;
        ks.x += kr * x[i].x; ks.y += kr * x[i].y; ks.z += kr * x[i].z; ks.w += kr * x[i].w;
      }
    }
    reinterpret_cast<float4*>(part)[tid] = ks;
    __syncthreads();
    float4 u = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p = 0; p < groups; ++p) {
      const float4 y = reinterpret_cast<const float4*>(part)[p * lanes + piece];
      u.x += y.x; u.y += y.y; u.z += y.z; u.w += y.w;
    }
    u.x = beta * (v.x - u.x); u.y = beta * (v.y - u.y); u.z = beta * (v.z - u.z); u.w = beta * (v.w - u.w);
    // ---- S <- S + k u^T, its product with the query
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int row = group + i * groups;
      if (row < dim) {
        const float kr = K[row], qr = Q[row];
        x[i].x += kr * u.x; x[i].y += kr * u.y; x[i].z += kr * u.z; x[i].w += kr * u.w;
        o.x += qr * x[i].x; o.y += qr * x[i].y; o.z += qr * x[i].z; o.w += qr * x[i].w;
      }
    }
    __syncthreads();                                         // the key products have been read
    reinterpret_cast<float4*>(part)[tid] = o;
    __syncthreads();
    if (group == 0 && col_ok) {
      o = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int p = 0; p < groups; ++p) {
        const float4 y = reinterpret_cast<const float4*>(part)[p * lanes + piece];
        o.x += y.x; o.y += y.y; o.z += y.z; o.w += y.w;
      }
      *reinterpret_cast<float4*>(out + (tok * heads + h) * (int64_t)vdim + col) = o;
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = group + i * groups;
    if (col_ok && row < dim) *reinterpret_cast<float4*>(S + (at0 + i * hop)) = x[i];
  }
}

// Sequences of at most `at_most` tokens: a long run meets six barriers a token here.  -> true when they went here: value channels in
// pieces of 16 bytes, key sizes up to 256.  Lanes across the value channels: as many as leave at most
// 8 rows per thread, but a whole 128-byte line at least.
template <typename T>
bool try_delta_step(float* out, const float* qkv, const void* beta_pre, int64_t beta_stride, const void* decay_pre,
                    int64_t decay_stride, int decay_per_head, const float* dt_bias, const float* a_log, float* state,
                    const int32_t* q_start, const int32_t* ctx_len, const int32_t* state_slot, int num_seqs, int heads,
                    int kv_heads, int dim, int vdim, int at_most, hipStream_t stream) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(state);
  if (vdim % 4 != 0 || (2 * kv_heads * dim) % 4 != 0 || at % 16 != 0 || dim > kStepThreads || num_seqs > 65535 || heads > 65535)
    return false;
  int lanes = 1;
  while (lanes < 32 && lanes * 4 < vdim && (lanes < 8 || dim * lanes * 2 <= 8 * kStepThreads)) lanes <<= 1;
  const int rows = (dim * lanes + kStepThreads - 1) / kStepThreads;
  const dim3 grid((unsigned)((vdim + lanes * 4 - 1) / (lanes * 4)), (unsigned)heads, (unsigned)num_seqs);
  const size_t bytes = sizeof(float) * ((3 * dim + 3) / 4 * 4 + kStepThreads * 4 + 8);
#define SWM_STEP(R)                                                                                                            \
  hipLaunchKernelGGL((delta_step_kernel<T, R>), grid, dim3(kStepThreads), bytes, stream, out, qkv, beta_pre, beta_stride,      \
                     decay_pre, decay_stride, decay_per_head, dt_bias, a_log, state, q_start, ctx_len, state_slot, heads,      \
                     kv_heads, dim, vdim, lanes, at_most)
  if (rows <= 4) SWM_STEP(4);
  else SWM_STEP(8);
#undef SWM_STEP
  return true;
}

bool delta_step(float* out, const float* qkv, const void* beta_pre, int64_t beta_stride, const void* decay_pre,
                int64_t decay_stride, int decay_per_head, const float* dt_bias, const float* a_log, float* state,
                const int32_t* q_start, const int32_t* ctx_len, const int32_t* state_slot, int num_seqs, int heads, int kv_heads,
                int dim, int vdim, int at_most, int act_dtype, hipStream_t stream) {
  bool taken = false;
  SWM_DISPATCH_ACT(act_dtype, taken = try_delta_step<T>(out, qkv, beta_pre, beta_stride, decay_pre, decay_stride, decay_per_head,
                                                        dt_bias, a_log, state, q_start, ctx_len, state_slot, num_seqs, heads,
                                                        kv_heads, dim, vdim, at_most, stream););
  return taken;
}

}  // namespace swm
