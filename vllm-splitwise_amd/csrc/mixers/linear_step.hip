// One decode step (or a few tokens) of linear attention:  S <- diag(a_t) S + k_t v_t^T,  o_t = S^T q_t  (S [dim, vdim] fp32), with a
// decay per key channel from a projection (gla.hip) or one per head (lightning.hip).
// What bounds it: the states, which are read and written once.  As in delta_step.hip a workgroup owns (sequence, head) and
// neighbouring value channels, thread (group, piece) the rows group, group + G, ... of 4 of them, so that a wave reads and writes
// the state in whole rows of 16-byte pieces, every load in flight before the first is used; queries, keys and decays are worked out
// meanwhile.  The rows' products with the query meet in LDS.
// Measured, norm and gate included, 61 sequences x 16 heads of 128 x 128 (128 MB of states read and written), a token each, us: gla
// 35.3 -> 28.4, lightning 74.1 -> 30.4, retention 68.3 -> 25.7 (before: by chunks of one, lightning's on the matrix cores, a lane holding
// a state's column 4 bytes at a time).  linear_plan.h says which steps come here.
#include "linear_walk.cuh"

namespace swm {

constexpr int kLinearThreads = 256;
enum LinearRule { kGla, kLightning, kRetention };

struct LinearDecay {
  const void* pre;                      // gla: projection [rows, heads * dim]; the others: fp32 [heads]
  int64_t stride;
  const float* bias;                    // gla, or NULL
  float inv_tau, q_scale;
};

// R: rows per thread (dim <= R * groups).  TQ, T: type of queries and keys, of values.
template <typename TQ, typename T, int RULE, int R>
__global__ __launch_bounds__(kLinearThreads) void linear_step_kernel(const LinearStep a, const LinearDecay decay, int lanes, int at_most) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int groups = kLinearThreads / lanes;                 // lanes: threads across the value channels, a power of two
  const int dim = a.dim, vdim = a.vdim;
  float* Q = lds;
  float* K = Q + dim;
  float* D = K + dim;
  float* part = lds + (3 * dim + 3) / 4 * 4;                 // [groups][lanes * 4]
  const int h = blockIdx.y, s = blockIdx.z;
  const int first = a.q_start[s], n = a.q_start[s + 1] - first;
  if (n <= 0 || n > at_most) return;                         // the whole workgroup
  const int tid = threadIdx.x, piece = tid % lanes, group = tid / lanes;
  const int col = (blockIdx.x * lanes + piece) * 4;
  const bool col_ok = col < vdim;                            // vdim is a multiple of 4
  float* S = a.state + ((int64_t)a.state_slot[s] * a.heads + h) * (int64_t)dim * vdim;     // uniform; 32-bit offsets from it
  const uint32_t at0 = (uint32_t)(group * vdim + col), hop = (uint32_t)(groups * vdim);
  const bool carried = a.ctx_len[s] > 0;
  float4 x[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = group + i * groups;
    x[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (carried && col_ok && row < dim) x[i] = *reinterpret_cast<const float4*>(S + (at0 + i * hop));
  }
  const float lam = RULE == kGla ? 0.0f : static_cast<const float*>(decay.pre)[h];
  for (int t = 0; t < n; ++t) {
    const int64_t tok = first + t, qk_at = tok * a.qk_stride + (int64_t)h * dim + tid;
    float qv = 0.0f, kv = 0.0f, g = lam;
    if (tid < dim) {                                         // dim <= 256
      qv = ld<TQ>(a.q, qk_at);
      kv = ld<TQ>(a.k, qk_at);
      if (RULE == kGla) {
        float z = ld<T>(decay.pre, tok * decay.stride + (int64_t)h * dim + tid);
        if (decay.bias != nullptr) z += decay.bias[h * dim + tid];
        qv *= decay.q_scale;
        g = expf(logsigmoidf_(z) * decay.inv_tau);
      } else if (RULE == kLightning) {
        qv = fast_siluf_(qv);
        kv = fast_siluf_(kv);
      }
    }
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (col_ok) {
      const int64_t v_at = tok * a.v_stride + (int64_t)h * vdim + col;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = ld<T>(a.v, v_at + j);
      if (RULE == kLightning) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = fast_siluf_(v[j]);
      }
    }
    if (tid < dim) {                                         // (the last token's have been read: a barrier lies between)
      Q[tid] = qv;
      K[tid] = kv;
      D[tid] = g;
    }
    __syncthreads();
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int row = group + i * groups;
      if (row < dim) {
        const float gr = RULE == kGla ? D[row] : lam, kr = K[row], qr = Q[row];
        x[i].x = gr * x[i].x + kr * v[0]; x[i].y = gr * x[i].y + kr * v[1];
        x[i].z = gr * x[i].z + kr * v[2]; x[i].w = gr * x[i].w + kr * v[3];
        o.x += qr * x[i].x; o.y += qr * x[i].y; o.z += qr * x[i].z; o.w += qr * x[i].w;
      }
    }
    reinterpret_cast<float4*>(part)[tid] = o;
    __syncthreads();
    if (group == 0 && col_ok) {
      o = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int p = 0; p < groups; ++p) {
        const float4 y = reinterpret_cast<const float4*>(part)[p * lanes + piece];
        o.x += y.x; o.y += y.y; o.z += y.z; o.w += y.w;
      }
      *reinterpret_cast<float4*>(a.out + (tok * a.heads + h) * (int64_t)vdim + col) = o;
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = group + i * groups;
    if (col_ok && row < dim) *reinterpret_cast<float4*>(S + (at0 + i * hop)) = x[i];
  }
}

// Sequences of at most `at_most` tokens.  -> true when they went here: value channels in pieces of 16 bytes, key sizes up to 256.
template <typename TQ, typename T, int RULE>
bool try_linear_step(const LinearStep& a, const LinearDecay& decay, int at_most, hipStream_t stream) {
  if (a.vdim % 4 != 0 || (reinterpret_cast<uintptr_t>(a.out) | reinterpret_cast<uintptr_t>(a.state)) % 16 != 0 ||
      a.dim > kLinearThreads || a.num_seqs > 65535 || a.heads > 65535 || (int64_t)a.dim * a.vdim >= 1ll << 31)
    return false;
  int lanes = 1;                                             // as many as leave at most 8 rows per thread, but a 128-byte line at least
  while (lanes < 32 && lanes * 4 < a.vdim && (lanes < 8 || a.dim * lanes * 2 <= 8 * kLinearThreads)) lanes <<= 1;
  const int rows = (a.dim * lanes + kLinearThreads - 1) / kLinearThreads;
  const dim3 grid((unsigned)((a.vdim + lanes * 4 - 1) / (lanes * 4)), (unsigned)a.heads, (unsigned)a.num_seqs);
  const size_t bytes = sizeof(float) * ((3 * a.dim + 3) / 4 * 4 + kLinearThreads * 4);
#define SWM_STEP(R) \
  hipLaunchKernelGGL((linear_step_kernel<TQ, T, RULE, R>), grid, dim3(kLinearThreads), bytes, stream, a, decay, lanes, at_most)
  if (rows <= 4) SWM_STEP(4);
  else SWM_STEP(8);
#undef SWM_STEP
  return true;
}

bool gla_step(const LinearStep& a, const void* decay_pre, int64_t decay_stride, const float* decay_bias, float inv_tau, float q_scale,
              int at_most, int act_dtype, hipStream_t stream) {
  const LinearDecay decay{decay_pre, decay_stride, decay_bias, inv_tau, q_scale};
  bool taken = false;
  SWM_DISPATCH_ACT(act_dtype, taken = (try_linear_step<T, T, kGla>(a, decay, at_most, stream)););
  return taken;
}

bool lightning_step(const LinearStep& a, const float* decay, bool silu, int at_most, int v_dtype, hipStream_t stream) {
  const LinearDecay d{decay, 0, nullptr, 0.0f, 1.0f};
  bool taken = false;
  if (silu) {
    SWM_DISPATCH_ACT(v_dtype, taken = (try_linear_step<T, T, kLightning>(a, d, at_most, stream)););
  } else {
    SWM_DISPATCH_ACT(v_dtype, taken = (try_linear_step<float, T, kRetention>(a, d, at_most, stream)););
  }
  return taken;
}

}  // namespace swm
