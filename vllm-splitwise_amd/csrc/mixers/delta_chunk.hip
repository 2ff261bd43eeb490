// The delta rule with a gate and ONE decay per head in chunks of 32 tokens, for steps that bring long runs:
//     S <- g_t S;  u_t = beta_t (v_t - S^T k_t);  S <- S + k_t u_t^T;  o_t = S^T q_t         (S [dim, vdim], fp32)
// With L_t = log g_1 + ... + log g_t inside a chunk (<= 0, so every ratio e^(L_t - L_s), s <= t, is at most 1) and S_0
// the state at the chunk's start, the chunk's u_t solve (I + A) U = W,  W = diag(beta) (V - diag(e^L) K S_0), with the strict
// lower triangle A[t, s] = beta_t e^(L_t - L_s) (k_t . k_s).  T = (I + A)^-1 does not depend on the state, so
//   a PROLOGUE, parallel over (chunk, key head), makes unit q and k and for each of the head's value heads beta, L, T by
//   forward substitution and P[t, s] = e^(L_t - L_s) (q_t . k_s) (s <= t);
//   the WALK goes through a sequence's chunks with   U = T W,   O = diag(e^L) Q S_0 + P U,
//   S_n = e^(L_n) S_0 + K^T diag(e^(L_n - L)) U,  fp32 products on the matrix cores, which is the recurrence with its sums
//   reordered.
//
// What bounds the walk is its chain: chunk after chunk, product after product.  A workgroup owns (sequence, head, 16 value
// channels); its wave b keeps the state's key coordinates 32 b .. 32 b + 31 in the accumulators of v_mfma_f32_16x16x4_f32
// (lane l: channel l % 16; element r of tile i: coordinate 32 b + 16 i + 4 (l / 16) + r), which is also how the B operand of the
// next product wants them.  Everything that a chunk brings comes straight from memory into the A operands' registers, asked
// for a chunk ahead; only the waves' shares of K S_0 and Q S_0 meet in LDS, behind the one barrier of a chunk.  Workgroups
// that read the same chunks (the channels of a head) have numbers 8 apart: one XCD, one L2.
// Measured, two prompts of 4324 tokens together, 16 heads on 8 of 128: prologue 321 us and walk 593 us with the chunk's operands
// multiplied out by the prologue, staged in LDS behind two barriers, and 32 channels per workgroup (128 workgroups); 69 and
// 233 us here.  Of the walk's 3.0 us a chunk 1.9 are its products, exchanges and waits alone (66 products of 32 cycles are 0.9),
// 0.6 the operands' way through the L1 and 0.5 their way from memory.
// L is summed in 64 bits: its differences are what counts, and where decays are strong 32 bits leave the end states an error of
// 0.5 - 1.3e-6 (1.3 - 1.5e-7 here, for the prologue's 69 us all the same).
// Rows of a last, shorter chunk are padded with beta = 0, k = 0, g = 1: they change nothing and are not stored.
#include "delta_step.h"
#include "mixers_common.cuh"

#include <algorithm>

namespace swm {

using f32x4 = __attribute__((ext_vector_type(4))) float;
using f32x16 = __attribute__((ext_vector_type(16))) float;
constexpr int kDcChunk = 32;
constexpr int kDcPrepThreads = 256;
constexpr int kDcShort = 16;             // tokens of a sequence that goes the decode kernel's way in a mixed step
constexpr int kDcChannels = 16;          // value channels of a walk's workgroup

// floats of one (chunk, key head) in the workspace: K | Q ([32][dp] each) | K^T [dp][32]
__host__ __device__ inline int64_t dc_keys_floats(int dp) { return 96 * (int64_t)dp; }
// ... and of one (chunk, value head): T | P ([32][32] each) | beta | e^L | e^(L_n - L) (32 each) | e^(L_n), padded
constexpr int kDcRecord = 2 * 1024 + 3 * 32 + 32;

__device__ __forceinline__ float dc_other_half(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float((threadIdx.x & 32) ? r[0] : r[1]);
}

template <typename T>
__global__ __launch_bounds__(kDcPrepThreads) void delta_chunk_prep_kernel(
    float* __restrict__ keys, float* __restrict__ records, const float* __restrict__ qkv, const void* __restrict__ beta_pre,
    int64_t beta_stride, const void* __restrict__ decay_pre, int64_t decay_stride, const float* __restrict__ dt_bias,
    const float* __restrict__ a_log, const int32_t* __restrict__ q_start, int num_seqs, int at_most, int heads, int kv_heads,
    int dim, int vdim, int dp) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int KS = dp + 4;                         // rows on 16 bytes
  float* Kn = lds;                               // [32][KS] unit keys
  float* Qn = Kn + kDcChunk * KS;                // [32][KS] unit queries times dim^-1/2
  float* red = Qn + kDcChunk * KS;               // [4 waves][2][4][64] quads: shares of K K^T and Q K^T; later A and L
  int seq = 0, tok0 = 0, before = 0;
  const int cn = find_run_piece(q_start, num_seqs, at_most, kDcChunk, blockIdx.x, &seq, &tok0, &before);
  if (cn <= 0) return;                           // the whole workgroup
  const int g = blockIdx.y, group = heads / kv_heads;
  const int64_t row0 = q_start[seq] + tok0;
  const int64_t row_w = 2 * (int64_t)kv_heads * dim + (int64_t)heads * vdim;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 31, hl = lane >> 5;
  // ---- the chunk's raw queries and keys into LDS (every load in flight at once), then unit length in place: 8 lanes a row
  for (int e = tid; e < kDcChunk * dp; e += kDcPrepThreads) {
    const int r = e / dp, i = e - r * dp;
    const bool in = r < cn && i < dim;
    const float* q = qkv + (row0 + r) * row_w + (int64_t)g * dim;
    Qn[r * KS + i] = in ? q[i] : 0.0f;
    Kn[r * KS + i] = in ? q[(int64_t)kv_heads * dim + i] : 0.0f;
  }
  __syncthreads();
  {
    const int r = tid >> 3, p = (tid & 7) * 4;
    float qq = 0.0f, kk = 0.0f;
    for (int i = p; i < dp; i += 32) {
      const float4 q = *reinterpret_cast<const float4*>(Qn + r * KS + i), k = *reinterpret_cast<const float4*>(Kn + r * KS + i);
      qq += q.x * q.x + q.y * q.y + q.z * q.z + q.w * q.w;
      kk += k.x * k.x + k.y * k.y + k.z * k.z + k.w * k.w;
    }
    qq = lanes_sum<8>(qq);
    kk = lanes_sum<8>(kk);
    const float qf = (1.0f / sqrtf((float)dim)) / sqrtf(qq + 1e-6f), kf = 1.0f / sqrtf(kk + 1e-6f);
    float* out = keys + ((int64_t)blockIdx.x * kv_heads + g) * dc_keys_floats(dp) + (int64_t)r * dp;
    for (int i = p; i < dp; i += 32) {
      float4 q = *reinterpret_cast<const float4*>(Qn + r * KS + i), k = *reinterpret_cast<const float4*>(Kn + r * KS + i);
      q.x *= qf; q.y *= qf; q.z *= qf; q.w *= qf;
      k.x *= kf; k.y *= kf; k.z *= kf; k.w *= kf;
      *reinterpret_cast<float4*>(Qn + r * KS + i) = q;
      *reinterpret_cast<float4*>(Kn + r * KS + i) = k;
      *reinterpret_cast<float4*>(out + i) = k;
      *reinterpret_cast<float4*>(out + 32 * (int64_t)dp + i) = q;
    }
  }
  __syncthreads();
  // ---- K^T for the walk; shares of K K^T and Q K^T (rows t, columns s), 32 coordinates at a time
  {
    float* kt = keys + ((int64_t)blockIdx.x * kv_heads + g) * dc_keys_floats(dp) + 64 * (int64_t)dp;
    for (int e = tid; e < dp * 8; e += kDcPrepThreads) {
      const int c = e >> 3, t = (e & 7) * 4;
      *reinterpret_cast<float4*>(kt + c * 32 + t) =
          make_float4(Kn[t * KS + c], Kn[(t + 1) * KS + c], Kn[(t + 2) * KS + c], Kn[(t + 3) * KS + c]);
    }
  }
  f32x16 kk, qk;
#pragma unroll
  for (int r = 0; r < 16; ++r) kk[r] = qk[r] = 0.0f;
  for (int b = wave; b * 32 < dp; b += kDcPrepThreads / 64) {
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const float4 k = *reinterpret_cast<const float4*>(Kn + li * KS + 32 * b + 8 * g4 + 4 * hl);
      const float4 q = *reinterpret_cast<const float4*>(Qn + li * KS + 32 * b + 8 * g4 + 4 * hl);
      kk = __builtin_amdgcn_mfma_f32_32x32x2f32(k.x, k.x, kk, 0, 0, 0);
      qk = __builtin_amdgcn_mfma_f32_32x32x2f32(q.x, k.x, qk, 0, 0, 0);
      kk = __builtin_amdgcn_mfma_f32_32x32x2f32(k.y, k.y, kk, 0, 0, 0);
      qk = __builtin_amdgcn_mfma_f32_32x32x2f32(q.y, k.y, qk, 0, 0, 0);
      kk = __builtin_amdgcn_mfma_f32_32x32x2f32(k.z, k.z, kk, 0, 0, 0);
      qk = __builtin_amdgcn_mfma_f32_32x32x2f32(q.z, k.z, qk, 0, 0, 0);
      kk = __builtin_amdgcn_mfma_f32_32x32x2f32(k.w, k.w, kk, 0, 0, 0);
      qk = __builtin_amdgcn_mfma_f32_32x32x2f32(q.w, k.w, qk, 0, 0, 0);
    }
  }
  float4* quads = reinterpret_cast<float4*>(red);
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) {
    quads[((wave * 2) * 4 + r4) * 64 + lane] = make_float4(kk[4 * r4], kk[4 * r4 + 1], kk[4 * r4 + 2], kk[4 * r4 + 3]);
    quads[((wave * 2 + 1) * 4 + r4) * 64 + lane] = make_float4(qk[4 * r4], qk[4 * r4 + 1], qk[4 * r4 + 2], qk[4 * r4 + 3]);
  }
  __syncthreads();
  // element r of a lane: t = 8 (r / 4) + 4 hl + r % 4, s = li
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) {
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), c = a;
#pragma unroll
    for (int w = 0; w < kDcPrepThreads / 64; ++w) {
      const float4 x = quads[((w * 2) * 4 + r4) * 64 + lane], y = quads[((w * 2 + 1) * 4 + r4) * 64 + lane];
      a.x += x.x; a.y += x.y; a.z += x.z; a.w += x.w;
      c.x += y.x; c.y += y.y; c.z += y.z; c.w += y.w;
    }
    kk[4 * r4] = a.x; kk[4 * r4 + 1] = a.y; kk[4 * r4 + 2] = a.z; kk[4 * r4 + 3] = a.w;
    qk[4 * r4] = c.x; qk[4 * r4 + 1] = c.y; qk[4 * r4 + 2] = c.z; qk[4 * r4 + 3] = c.w;
  }
  __syncthreads();
  // ---- a wave per value head of this key head
  float* A = red + wave * (kDcChunk * 36 + 96);  // [32][36]: row t, its even columns, then its odd ones
  double* Ls = reinterpret_cast<double*>(A + kDcChunk * 36);  // [32] running sums of the log decays
  float* Bs = A + kDcChunk * 36 + 64;            // [32] beta
  for (int m = wave; m < group; m += kDcPrepThreads / 64) {
    const int h = g * group + m;
    float* rec = records + ((int64_t)blockIdx.x * heads + h) * kDcRecord;
    float beta = 0.0f;
    double L = 0.0;                              // of token li, in both halves
    if (li < cn) {
      beta = sigmoidf_(ld<T>(beta_pre, (row0 + li) * beta_stride + h));
      L = -expf(a_log[h]) * softplusf_(ld<T>(decay_pre, (row0 + li) * decay_stride + h) + dt_bias[h]);
    }
#pragma unroll
    for (int step = 1; step < 32; step <<= 1) {
      const double o = __shfl_up(L, step, 32);
      if (li >= step) L += o;
    }
    const double Ln = __shfl(L, 31, 32);
    if (hl == 0) {
      Ls[li] = L;
      Bs[li] = beta;
      rec[2048 + li] = beta;
      rec[2048 + 32 + li] = expf((float)L);
      rec[2048 + 64 + li] = expf((float)(Ln - L));
      if (li == 0) rec[2048 + 96] = expf((float)Ln);
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int t = 8 * (r / 4) + 4 * hl + r % 4;
      const float ratio = li <= t ? expf((float)(Ls[t] - L)) : 0.0f;
      A[t * 36 + (li & 1) * 16 + (li >> 1)] = li < t ? Bs[t] * ratio * kk[r] : 0.0f;
      rec[1024 + t * 32 + li] = ratio * qk[r];
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    // T = (I + A)^-1 row by row: T[t, :] = e_t - sum_{s < t} A[t, s] T[s, :].  Lane li holds column li, the half hl its rows of
    // that parity.
    float col[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) col[i] = 0.0f;
#pragma unroll
    for (int t = 0; t < kDcChunk; ++t) {
      float p0 = 0.0f, p1 = 0.0f;
#pragma unroll
      for (int i4 = 0; i4 < (t + 7) / 8; ++i4) {             // columns 2 i + hl < t (A is zero from the diagonal on)
        const float4 x = *reinterpret_cast<const float4*>(A + t * 36 + hl * 16 + 4 * i4);
        p0 += x.x * col[4 * i4] + x.y * col[4 * i4 + 1];
        p1 += x.z * col[4 * i4 + 2] + x.w * col[4 * i4 + 3];
      }
      const float sum = p0 + p1;
      const float v = (t == li ? 1.0f : 0.0f) - (sum + dc_other_half(sum));
      if ((t & 1) == hl) {
        col[t / 2] = v;
        rec[t * 32 + li] = v;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// What a chunk brings to a wave, in the layouts of the A operands (16 x 4: lane l is row l % 16, reduction index l / 16)
struct DcOperands {
  f32x4 k[2][2], q[2][2];                        // [16 tokens][16 coordinates]: token l % 16, coordinates 4 (l / 16) ..
  f32x4 kt[2][2];                                // [16 coordinates][16 tokens]: coordinate l % 16, tokens 4 (l / 16) ..
  f32x4 t[3], p[3];                              // tiles (0, 0), (1, 0), (1, 1) of T and P: row l % 16, columns 4 (l / 16) ..
  f32x4 v[2], beta[2], el[2], tail[2];           // tokens 16 i + 4 (l / 16) .. of this lane's channel / of the head
  float keep;                                    // e^(L_n)
};

template <int NDB>
__global__ __launch_bounds__(64 * NDB) void delta_chunk_kernel(
    float* __restrict__ out, const float* __restrict__ keys, const float* __restrict__ records, const float* __restrict__ qkv,
    float* __restrict__ state, const int32_t* __restrict__ q_start, const int32_t* __restrict__ ctx_len,
    const int32_t* __restrict__ state_slot, int num_seqs, int at_most, int64_t runs, int heads, int kv_heads, int dim, int vdim) {
  __shared__ f32x4 red[2][2][NDB][2][64];        // [chunk parity][K S_0 | Q S_0][wave][token tile][lane]
  constexpr int DP = NDB * 32;
  const int vblocks = (vdim + kDcChannels - 1) / kDcChannels;
  const int unit = (blockIdx.x >> 3) / vblocks * 8 + (blockIdx.x & 7), vb = (blockIdx.x >> 3) % vblocks;
  const int run = unit / heads, h = unit - run * heads, g = h / (heads / kv_heads);
  int seq = 0, tok0 = 0, chunk0 = 0;             // chunk0: this sequence's first chunk among the step's
  const int n = run < runs ? find_run_piece(q_start, num_seqs, at_most, 1 << 30, run, &seq, &tok0, &chunk0) : 0;
  if (n <= 0) return;                            // the whole workgroup
  const int b = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, gq = lane >> 4;
  const int64_t row0 = q_start[seq];
  const int vc = vb * kDcChannels + li;          // this lane's value channel
  const bool vc_ok = vc < vdim;
  float* sp = state + ((int64_t)state_slot[seq] * heads + h) * (int64_t)dim * vdim;
  f32x4 S[2];
  const bool fresh = ctx_len[seq] == 0;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int c = 32 * b + 16 * i + 4 * gq + r;
      S[i][r] = (!fresh && vc_ok && c < dim) ? sp[(int64_t)c * vdim + vc] : 0.0f;
    }
  const int64_t row_w = 2 * (int64_t)kv_heads * dim + (int64_t)heads * vdim;
  const float* vsrc = qkv + row0 * row_w + 2 * (int64_t)kv_heads * dim + (int64_t)h * vdim + (vc_ok ? vc : vdim - 1);
  const int chunks = (n + kDcChunk - 1) / kDcChunk;
  auto fetch = [&](DcOperands& x, int ci) {
    const float* kp = keys + ((int64_t)(chunk0 + ci) * kv_heads + g) * dc_keys_floats(DP);
    const float* rec = records + ((int64_t)(chunk0 + ci) * heads + h) * kDcRecord;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float* kr = kp + (16 * i + li) * DP + 32 * b + 16 * j + 4 * gq;
        x.k[i][j] = *reinterpret_cast<const f32x4*>(kr);
        x.q[i][j] = *reinterpret_cast<const f32x4*>(kr + 32 * DP);
        x.kt[i][j] = *reinterpret_cast<const f32x4*>(kp + 64 * DP + (32 * b + 16 * i + li) * 32 + 16 * j + 4 * gq);
      }
      x.beta[i] = *reinterpret_cast<const f32x4*>(rec + 2048 + 16 * i + 4 * gq);
      x.el[i] = *reinterpret_cast<const f32x4*>(rec + 2048 + 32 + 16 * i + 4 * gq);
      x.tail[i] = *reinterpret_cast<const f32x4*>(rec + 2048 + 64 + 16 * i + 4 * gq);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x.v[i][r] = vsrc[min(ci * kDcChunk + 16 * i + 4 * gq + r, n - 1) * row_w];
      }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const float* tile = rec + (i == 0 ? 0 : 16 * 32) + (i == 2 ? 16 : 0) + li * 32 + 4 * gq;
      x.t[i] = *reinterpret_cast<const f32x4*>(tile);
      x.p[i] = *reinterpret_cast<const f32x4*>(tile + 1024);
    }
    x.keep = rec[2048 + 96];
  };
  // The outputs of a chunk wait for its shares of Q S_0, which meet in LDS behind the NEXT chunk's barrier: the wave that
  // finishes token tile i keeps P U and e^L until then.
  f32x4 pu[2], pel[2];
  auto finish = [&](int ci, const f32x4 (&own)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if ((2 * ci + i) % NDB != b) continue;     // wave-uniform
      f32x4 o = own[i];
      if (NDB > 1) {
        f32x4 part[NDB];
#pragma unroll
        for (int w = 0; w < NDB; ++w) part[w] = red[ci & 1][1][w][i][lane];
        o = part[0];
#pragma unroll
        for (int w = 1; w < NDB; ++w) o += part[w];
      }
      o = o * pel[i] + pu[i];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = ci * kDcChunk + 16 * i + 4 * gq + r;
        if (vc_ok && t < n) out[((row0 + t) * heads + h) * (int64_t)vdim + vc] = o[r];
      }
    }
  };
  f32x4 qs[2];
  auto chunk = [&](const DcOperands& x, int ci) {
    const int buf = ci & 1;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    // ---- this wave's share of K S_0, which everything waits for
    f32x4 ks[2] = {zero, zero}, part[NDB][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i) ks[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[i][j][r], S[j][r], ks[i], 0, 0, 0);
    if (NDB > 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i) red[buf][0][b][i][lane] = ks[i];
      __syncthreads();                           // (two buffers: nobody is more than a chunk ahead of a reader)
#pragma unroll
      for (int w = 0; w < NDB; ++w)
#pragma unroll
        for (int i = 0; i < 2; ++i) part[w][i] = red[buf][0][w][i][lane];
    }
    if (ci > 0) finish(ci - 1, qs);
    __builtin_amdgcn_sched_barrier(0);
    // ---- ... and of Q S_0 while the others' arrive
#pragma unroll
    for (int i = 0; i < 2; ++i) qs[i] = zero;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i) qs[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[i][j][r], S[j][r], qs[i], 0, 0, 0);
    if (NDB > 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        ks[i] = part[0][i];
#pragma unroll
        for (int w = 1; w < NDB; ++w) ks[i] += part[w][i];
      }
    }
    // ---- W = diag(beta) (V - diag(e^L) K S_0), U = T W: element r of tile i is token 16 i + 4 gq + r
    f32x4 w[2], u[2] = {zero, zero};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      w[i] = x.beta[i] * (x.v[i] - x.el[i] * ks[i]);
#pragma unroll
      for (int r = 0; r < 4; ++r)                // (the padding read some other token's value)
        if (ci * kDcChunk + 16 * i + 4 * gq + r >= n) w[i][r] = 0.0f;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      u[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.t[0][r], w[0][r], u[0], 0, 0, 0);
      u[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.t[1][r], w[0][r], u[1], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) u[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.t[2][r], w[1][r], u[1], 0, 0, 0);
    if (NDB > 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i) red[buf][1][b][i][lane] = qs[i];
    }
    // ---- S <- e^(L_n) S + K^T diag(e^(L_n - L)) U
    f32x4 ut[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      ut[i] = x.tail[i] * u[i];
      S[i] *= x.keep;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i) S[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kt[i][j][r], ut[j][r], S[i], 0, 0, 0);
    // ---- O = diag(e^L) Q S_0 + P U, the token tiles by different waves, in turn
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if ((2 * ci + i) % NDB != b) continue;     // wave-uniform
      pel[i] = x.el[i];
      pu[i] = zero;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pu[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.p[i][r], u[0][r], pu[i], 0, 0, 0);
        if (i == 1) pu[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.p[2][r], u[1][r], pu[i], 0, 0, 0);
      }
    }
  };
  // (the barriers of the schedule keep a chunk's loads in front of the products of the chunk before it)
  if constexpr (NDB <= 4) {
    DcOperands x0, x1;
    fetch(x0, 0);
#pragma unroll 1
    for (int ci = 0; ci < chunks; ci += 2) {     // uniform over the workgroup: every wave meets every barrier
      fetch(x1, min(ci + 1, chunks - 1));
      __builtin_amdgcn_sched_barrier(0);
      chunk(x0, ci);
      if (ci + 1 >= chunks) break;
      fetch(x0, min(ci + 2, chunks - 1));
      __builtin_amdgcn_sched_barrier(0);
      chunk(x1, ci + 1);
    }
  } else {                                       // more than a wave per SIMD: no registers for a chunk ahead
    DcOperands x;
#pragma unroll 1
    for (int ci = 0; ci < chunks; ++ci) {
      fetch(x, ci);
      chunk(x, ci);
    }
  }
  if (NDB > 1) __syncthreads();
  finish(chunks - 1, qs);
  if (vc_ok) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = 32 * b + 16 * i + 4 * gq + r;
        if (c < dim) sp[(int64_t)c * vdim + vc] = S[i][r];
      }
  }
}

template <typename K>
inline hipError_t dc_allow_lds(K kernel, size_t bytes) {
  if (bytes <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

template <int NDB>
int launch_delta_chunk(float* out, const float* keys, const float* records, const float* qkv, float* state, const int32_t* q_start,
                       const int32_t* ctx_len, const int32_t* state_slot, int num_seqs, int at_most, int64_t runs, int heads,
                       int kv_heads, int dim, int vdim, hipStream_t stream) {
  const int64_t units = (runs * heads + 7) / 8 * 8, groups = units * ((vdim + kDcChannels - 1) / kDcChannels);
  SW_CHECK_ARG(groups < (1ll << 31), "gated_delta_chunked: too many sequences and heads");
  hipLaunchKernelGGL(delta_chunk_kernel<NDB>, dim3((unsigned)groups), dim3(64 * NDB), 0, stream, out, keys, records, qkv, state,
                     q_start, ctx_len, state_slot, num_seqs, at_most, runs, heads, kv_heads, dim, vdim);
  SW_CHECK_LAUNCH();
  return SW_OK;
}

}  // namespace swm

extern "C" {

int64_t swm_gated_delta_chunked_workspace_floats(int64_t rows, int num_seqs, int heads, int dim, int vdim) {
  const int dp = (dim + 31) / 32 * 32;
  (void)vdim;
  return (rows / swm::kDcChunk + num_seqs) * heads * (swm::dc_keys_floats(dp) + swm::kDcRecord);     // as many key heads at most
}

int swm_gated_delta_chunked(float* out, const float* qkv, const void* beta_pre, int64_t beta_stride,
                            const void* decay_pre, int64_t decay_stride, const float* dt_bias, const float* a_log,
                            float* state, const int32_t* q_start, const int32_t* ctx_len, const int32_t* state_slot,
                            int64_t rows, int num_seqs, int heads, int kv_heads, int dim, int vdim, float* workspace,
                            int act_dtype, void* stream) {
  using namespace swm;
  if (num_seqs == 0 || rows == 0) return SW_OK;
  SW_CHECK_ARG(act_ok(act_dtype), "gated_delta_chunked: unsupported dtype %d", act_dtype);
  SW_CHECK_ARG(heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && dim <= 224 && vdim > 0 &&
                   workspace != nullptr && rows < (1ll << 31),
               "gated_delta_chunked: heads %d, kv heads %d, key size %d (up to 224), value size %d", heads, kv_heads, dim,
               vdim);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int ndb = (dim + 31) / 32, dp = ndb * 32;
  // Decoding sequences beside a portion take the decode kernel: their states are read and written in whole rows there, in 64-byte
  // pieces here, and they need no 32-row record.  Not worth the launch where most sequences are long.  (us a call, 12 heads of 96, a
  // portion of 100 tokens beside 60 / 250 decoding sequences: 186 / 1046 all in chunks, 61 / 104 so)
  const bool mixed = num_seqs >= 12 && rows < 128 * (int64_t)num_seqs &&
                     delta_step(out, qkv, beta_pre, beta_stride, decay_pre, decay_stride, 1, dt_bias, a_log, state, q_start, ctx_len,
                                state_slot, num_seqs, heads, kv_heads, dim, vdim, kDcShort, act_dtype, s);
  SW_CHECK_LAUNCH();
  const int at_most = mixed ? kDcShort : 0;
  const int64_t runs = mixed ? std::min<int64_t>(num_seqs, rows / (kDcShort + 1)) : num_seqs;
  if (runs == 0) return SW_OK;
  const int64_t chunks = rows / kDcChunk + runs;                // an upper bound: surplus workgroups leave at once
  float* keys = workspace;
  float* records = workspace + chunks * kv_heads * dc_keys_floats(dp);
  const size_t prep_lds = sizeof(float) * (2 * (size_t)kDcChunk * (dp + 4) + 4 * 2 * 4 * 64 * 4);
  SWM_DISPATCH_ACT(act_dtype, SW_CHECK_HIP(dc_allow_lds(delta_chunk_prep_kernel<T>, prep_lds)););
  SWM_DISPATCH_ACT(act_dtype, hipLaunchKernelGGL(delta_chunk_prep_kernel<T>, dim3((unsigned)chunks, (unsigned)kv_heads),
                                                 dim3(kDcPrepThreads), prep_lds, s, keys, records, qkv, beta_pre, beta_stride,
                                                 decay_pre, decay_stride, dt_bias, a_log, q_start, num_seqs, at_most, heads,
                                                 kv_heads, dim, vdim, dp););
  SW_CHECK_LAUNCH();
#define SWM_DC_CASE(N)                                                                                                       \
  case N:                                                                                                                    \
    return launch_delta_chunk<N>(out, keys, records, qkv, state, q_start, ctx_len, state_slot, num_seqs, at_most, runs, heads, \
                                 kv_heads, dim, vdim, s);
  switch (ndb) {
    SWM_DC_CASE(1)
    SWM_DC_CASE(2)
    SWM_DC_CASE(3)
    SWM_DC_CASE(4)
    SWM_DC_CASE(5)
    SWM_DC_CASE(6)
    default: SWM_DC_CASE(7)
  }
#undef SWM_DC_CASE
}

}  // extern "C"
