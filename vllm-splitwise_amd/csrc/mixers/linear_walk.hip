// Linear attention over long runs:  S_t = diag(a_t) S_(t-1) + k_t v_t^T,  o_t = S_t^T q_t,  S [key size, value size] fp32 carried
// per sequence, with a decay per head and key channel (gla.hip) or one constant per head (lightning.hip), in chunks of 32 tokens:
//     O = A V + Q~ S_0,   S_n = diag(d) S_0 + K~^T V,
//     Q~_i = q_i a_1 .. a_i,   K~_j = k_j a_(j+1) .. a_n,   d = a_1 .. a_n,   A[i, j] = sum_c q_ic k_jc a_(j+1) .. a_i   (j <= i)
// A PROLOGUE, parallel over (chunk, head), writes Q~, K~^T, d and A; a WALK goes through a sequence's chunks.
//
// Every factor above is a product of decays and at most 1, so nothing overflows however strong they are.  Only A, as a matrix
// product, needs its decays taken apart: between the chunk's halves of 16 tokens at the border, where both parts are again
// at most 1; inside a half as p_i / p_j with p the half's running products.  A half in which some channel's product falls
// below e^-kLwSafeLog has its 16 x 16 weights worked out on the vector units instead, with the decays multiplied up token by token.
// Products are exponentials of running SUMS of log a, from the half's border towards the token: a decay near 1 (most are) has
// few significant digits left once it is rounded to a float, and over thousands of tokens the state would show it.
//
// The walk's only chain is the state itself, an accumulation: a workgroup owns (sequence, head, 16 value channels) and has two waves
// per 32 key coordinates.  One keeps the STATE's coordinates 32 b .. 32 b + 31 in the accumulators of v_mfma_f32_16x16x4_f32 (lane l:
// channel l % 16; element r of tile i: coordinate 32 b + 16 i + 4 (l / 16) + r), in the layout that the B operand of the next
// product wants; one makes the OUTPUTS, with the state from LDS, beside the state's next chunk.  Operands come straight from memory
// into registers, two chunks ahead, from a workspace that has them in the lanes' order, so that every load is a whole kilobyte; one
// wave reads and widens the values for all.  The shares of Q~ S_0 meet in LDS behind the one barrier of a chunk.  Workgroups that
// read the same chunks (the channels of a head) have numbers 8 apart: one XCD, one L2.
// The chain of a long run of few heads leaves the rest of the GPU idle.  Such a run is cut into segments (linear_plan.h): a launch
// of their own works out every segment's end from nothing, without outputs, exchange or barrier, and the walk then begins each
// segment at the end of the one in front of it, S = D S' + local end after local end, D the segment's products of decays.
//
// Measured, two prompts of 4324 tokens together, 16 heads of 128, a decay per key channel: 676 + 20 us in segments of 128 tokens
// taken twice, from nothing and from their true states, with a scan between (560 workgroups on 512 places: the second round
// nearly empty); 46 us prologue and 136 us walk with one wave per 32 coordinates for state and outputs, operands in rows and stores
// under a condition; 45 and 78 here.  Of the walk's 1.0 us a chunk the products are 0.5 (38 of 32 cycles), the rest the exchange and
// its barrier, and 37 KB of operands through the L1.  The prologue's bytes (135 MB) would take
// 27; the rest is vector work: the exponentials (52 us with expf and divisions), and 48 row addresses, uniform over the wave, that do
// not fit the scalar registers and travel through the lanes of vector registers (226 of them spilled).
// Relative error of the end states against 64 bits: 1.3e-7 here, 2.2e-7 in segments taken twice.
// One run of 16000 tokens, 4 heads of 128, decays per channel / per head: 448 / 468 us in one piece, 138 / 140 in 8 segments (415 /
// 300 in segments of 128 tokens); of 32000 tokens, 16 heads: 1120 and 1015 in 2.
#include "linear_walk.cuh"

#include <type_traits>

namespace swm {

using f32x4 = __attribute__((ext_vector_type(4))) float;
constexpr int kLwThreads = 256;
constexpr int kLwChannels = 16;
constexpr float kLwSafeLog = 12.0f;

// e^x, x <= 0: the hardware's 2^x, which is good to its last place, with the rounding of x log2(e) put back; half of expf's
// instructions, which allow for overflow and results below 2^-126 (0 here).  The rounding is below 2^-16 wherever 2^x is not 0.  It is
// bounded because a gate that overflowed is a log decay of -inf, of which it would be inf - inf: 0 as expf's, and NaN stays NaN.
__device__ __forceinline__ float exp_of_sum(float x) {
  const float y = x * 1.44269504f, rest = fmaf(x, 1.44269504f, -y) + x * 1.92596299e-8f;
  const float e = __builtin_amdgcn_exp2f(y);
  return fmaf(e, __builtin_amdgcn_fmed3f(rest, -1.0f, 1.0f) * 0.69314718f, e);
}
// 1 / p, e^-kLwSafeLog <= p <= 1
__device__ __forceinline__ float reciprocal_of(float p) {
  const float r = __builtin_amdgcn_rcpf(p);
  return fmaf(fmaf(-p, r, 1.0f), r, r);
}

// log(sigmoid(x)) = min(x, 0) - log(1 + t), t = e^-|x|, the logarithm on the hardware's log2 with the rounding of 1 + t put back:
// largest relative error over [-30, 30] 2.7e-7 (with log1pf 1.3e-7), root mean square 3.8e-8 (2.6e-8), a quarter of the instructions.
// The results do not show it: over runs of 40 to 3000 tokens, 4 to 16 heads of 64 to 128, tau 1 to 16, outputs are 1.5 - 2.1e-7 and
// end states 1.0 - 1.9e-7 from 64 bits with either (2.4 - 3.4e-7 and 1.2 - 2.8e-7 before this file); with log1pf prologue and walk
// of the step above take 128 us together instead of 111.
__device__ __forceinline__ float log_sigmoid(float x) {
  const float t = exp_of_sum(-fabsf(x)), u = 1.0f + t;
  return fminf(x, 0.0f) - (0.69314718055994531f * __builtin_amdgcn_logf(u) + (t - (u - 1.0f)) * __builtin_amdgcn_rcpf(u));
}

// The workspace holds the operands of the walk's products in the order in which its lanes read them: FRAGMENTS of 64 quads, one a
// lane, of a 16 x 16 tile.  Floats of one (chunk, head): Q~ by [32 coordinates][16 tokens][16 coordinates] | K~^T by
// [32 coordinates][16 coordinates][16 tokens] | d [dp] | tiles (0, 0), (1, 0), (1, 1) of A, in
// the place of four
__host__ __device__ inline int64_t lw_record(int dp) { return 65 * (int64_t)dp + 1024; }
// quad of coordinates c .. c + 3 of token t among Q~, of tokens t .. t + 3 of coordinate c among K~^T
__device__ __forceinline__ int lw_q_quad(int t, int c) { return (c >> 5) * 256 + (t >> 4) * 128 + ((c >> 4) & 1) * 64 + ((c & 15) >> 2) * 16 + (t & 15); }
__device__ __forceinline__ int lw_k_quad(int t, int c) { return (c >> 4) * 128 + (t >> 4) * 64 + ((t & 15) >> 2) * 16 + (c & 15); }

// the 16 x 16 weights of rows Y (keys) against rows X (queries): element r of lane l is query l % 16, key 4 (l / 16) + r
__device__ __forceinline__ f32x4 lw_block(const float* X, const float* Y, int KS, int dp) {
  const int lane = threadIdx.x & 63, li = lane & 15, gq = lane >> 4;
  f32x4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;
  for (int c = 4 * gq; c < dp; c += 32) {
    const float4 x = *reinterpret_cast<const float4*>(X + li * KS + c), y = *reinterpret_cast<const float4*>(Y + li * KS + c);
    const float4 x1 = *reinterpret_cast<const float4*>(X + li * KS + c + 16), y1 = *reinterpret_cast<const float4*>(Y + li * KS + c + 16);
    s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(y.x, x.x, s0, 0, 0, 0);
    s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(y1.x, x1.x, s1, 0, 0, 0);
    s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(y.y, x.y, s0, 0, 0, 0);
    s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(y1.y, x1.y, s1, 0, 0, 0);
    s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(y.z, x.z, s0, 0, 0, 0);
    s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(y1.z, x1.z, s1, 0, 0, 0);
    s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(y.w, x.w, s0, 0, 0, 0);
    s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(y1.w, x1.w, s1, 0, 0, 0);
  }
  return s0 + s1;
}

// 8 neighbouring numbers of row `row`, zeros where the row or the channels are not there
template <typename T>
__device__ __forceinline__ void lw_load8(float (&x)[8], const void* p, int64_t at, int c, int dim, bool in, bool vec) {
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = 0.0f;
  if (!in) return;
  if (vec && c + 8 <= dim) {
    if constexpr (sizeof(typename Conv<T>::store_t) == 2) {
      ld_vec<T, 8>(x, p, at + c);
    } else {
      float lo[4], hi[4];
      ld_vec<T, 4>(lo, p, at + c);
      ld_vec<T, 4>(hi, p, at + c + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = lo[j], x[4 + j] = hi[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (c + j < dim) x[j] = ld<T>(p, at + c + j);
  }
}
__device__ __forceinline__ void lw_put8(float* p, const float (&x)[8]) {
  *reinterpret_cast<float4*>(p) = make_float4(x[0], x[1], x[2], x[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(x[4], x[5], x[6], x[7]);
}

template <typename T>
__global__ __launch_bounds__(kLwThreads, 3) void gla_walk_prep_kernel(const LinearStep a, int at_most, const void* __restrict__ decay_pre,
                                                                   int64_t decay_stride, const float* __restrict__ decay_bias,
                                                                   float inv_tau, float q_scale, int dp) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int KS = dp + 4;
  float* Qs = lds;                               // [32][KS] queries times p
  float* Ks = Qs + kLwChunk * KS;                // [32][KS] keys divided by p
  float* Ko = Ks + kLwChunk * KS;                // [16][KS] the first half's keys carried to its end
  float* total = Ko + 16 * KS;                   // [2][dp] the halves' sums of log a
  float* ahead = total + 2 * dp;                 // [dp] the first half's product of decays
  int* unsafe = reinterpret_cast<int*>(ahead + dp);                      // [2]
  int seq = 0, tok0 = 0, before = 0;
  const int cn = find_run_piece(a.q_start, a.num_seqs, at_most, kLwChunk, blockIdx.x, &seq, &tok0, &before);
  if (cn <= 0) return;                           // the whole workgroup
  const int h = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int64_t row0 = a.q_start[seq] + tok0;
  float* rec = a.workspace + ((int64_t)blockIdx.x * a.heads + h) * lw_record(dp);
  float4* Qg = reinterpret_cast<float4*>(rec);
  float4* Kt = reinterpret_cast<float4*>(rec + 32 * (int64_t)dp);
  float* keep = rec + 64 * (int64_t)dp;
  float* A = rec + 65 * (int64_t)dp;
  if (tid < 2) unsafe[tid] = 0;
  __syncthreads();
  // ---- a thread per (channel, half), its 16 tokens in registers; key sizes beyond 128 take a second round
  const int half = __builtin_amdgcn_readfirstlane(tid / (kLwThreads / 2));
  for (int c0 = 0; c0 < dp; c0 += kLwThreads / 2) {
    const int c = c0 + tid % (kLwThreads / 2);
    const bool mine = c < dp, in = c < a.dim;
    float k[16], q[16], g[16], sum = 0.0f;
    if (mine) {
      const int col = h * a.dim + min(c, a.dim - 1);
      const float bias = decay_bias != nullptr ? decay_bias[col] : 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {             // (the rows' addresses are uniform over the wave)
        const int64_t row = row0 + min(16 * half + i, cn - 1);
        k[i] = ld<T>(static_cast<const typename Conv<T>::store_t*>(a.k) + row * a.qk_stride, col);
        q[i] = ld<T>(static_cast<const typename Conv<T>::store_t*>(a.q) + row * a.qk_stride, col);
        g[i] = ld<T>(static_cast<const typename Conv<T>::store_t*>(decay_pre) + row * decay_stride, col);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const bool there = in && 16 * half + i < cn;         // rows beyond the chunk: no key, no decay
        k[i] = there ? k[i] : 0.0f;
        q[i] = there ? q[i] * q_scale : 0.0f;
        g[i] = there ? log_sigmoid(g[i] + bias) * inv_tau : 0.0f;
        sum += g[i];
      }
      total[half * dp + c] = sum;
      if (!(sum >= -kLwSafeLog)) unsafe[half] = 1;
    }
    __syncthreads();
    if (mine) {                                  // (in a half that is not safe the keys may overflow: they are put back below)
      const float after = half ? 1.0f : exp_of_sum(total[dp + c]);
      if (half == 0) keep[c] = exp_of_sum(total[c] + total[dp + c]);
      if (half == 1) ahead[c] = exp_of_sum(total[c]);
      float run = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {             // towards the half's end: queries, and keys for the half's own weights
        run += g[i];
        const float p = exp_of_sum(run);
        q[i] *= p;
        Qs[(16 * half + i) * KS + c] = q[i];
        Ks[(16 * half + i) * KS + c] = k[i] * reciprocal_of(p);
      }
      run = 0.0f;
#pragma unroll
      for (int i = 15; i >= 0; --i) {            // towards its start: keys carried to the end
        k[i] *= exp_of_sum(run);
        run += g[i];
        if (half == 0) Ko[i * KS + c] = k[i];
      }
#pragma unroll
      for (int i = 0; i < 16; i += 4)
        Kt[lw_k_quad(16 * half + i, c)] =
            make_float4(k[i] * after, k[i + 1] * after, k[i + 2] * after, k[i + 3] * after);
    }
  }
  __syncthreads();
  for (int e = tid; e < 8 * dp; e += kLwThreads) {           // queries carried from the chunk's start
    const int t = (e >> 6 & 1) * 16 + (e & 15), c = (e >> 7) * 16 + (e >> 4 & 3) * 4;
    float4 q = *reinterpret_cast<const float4*>(Qs + t * KS + c);
    if (t >= 16) {
      const float4 f = *reinterpret_cast<const float4*>(ahead + c);
      q.x *= f.x; q.y *= f.y; q.z *= f.z; q.w *= f.w;
    }
    Qg[lw_q_quad(t, c)] = q;
  }
  // ---- the chunk's weights: wave 0 and 1 the halves' own, wave 2 the second half's on the first
  const int li = lane & 15, gq = lane >> 4;
  if (wave < 3 && !(wave < 2 && unsafe[wave] != 0)) {
    const int bi = wave == 0 ? 0 : 1, bj = wave == 1 ? 1 : 0;
    const f32x4 w = lw_block(Qs + bi * 16 * KS, wave == 2 ? Ko : Ks + bj * 16 * KS, KS, dp);
    f32x4 a;
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = bi > bj || 4 * gq + r <= li ? w[r] : 0.0f;
    reinterpret_cast<f32x4*>(A)[(bi + bj) * 64 + lane] = a;
  }
  if (unsafe[0] == 0 && unsafe[1] == 0) return;  // uniform over the workgroup
  __syncthreads();
  for (int e = tid; e < kLwChunk * dp; e += kLwThreads) {    // the decays themselves in Qs, the keys as they are in Ks
    const int r = e / dp, c = e - r * dp;
    float d = 1.0f, k = 0.0f;
    if (r < cn && c < a.dim) {
      const int64_t col = (int64_t)h * a.dim + c;
      const float z = ld<T>(decay_pre, (row0 + r) * decay_stride + col) + (decay_bias != nullptr ? decay_bias[col] : 0.0f);
      d = expf(log_sigmoid(z) * inv_tau);
      k = ld<T>(a.k, (row0 + r) * a.qk_stride + col);
    }
    Qs[r * KS + c] = d;
    Ks[r * KS + c] = k;
  }
  __syncthreads();
  for (int part = 0; part < 2; ++part) {
    if (unsafe[part] == 0) continue;             // uniform over the workgroup
    // 16 lanes share a key's channels; from the key on, its weight for one query after the other
    const int j = 16 * part + (tid >> 4);
    float sum[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) sum[i] = 0.0f;
    for (int c = tid & 15; c < a.dim; c += 16) {
      float kd = Ks[j * KS + c];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = 16 * part + i;
        if (t < j || t >= cn) continue;
        if (t > j) kd *= Qs[t * KS + c];
        sum[i] += ld<T>(a.q, (row0 + t) * a.qk_stride + (int64_t)h * a.dim + c) * q_scale * kd;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float w = lanes_sum<16>(sum[i]);
      if ((tid & 15) == i) A[part * 512 + (((j & 15) >> 2) * 16 + i) * 4 + (j & 3)] = w;      // (0 where j > i)
    }
  }
}

// vec: rows of q and k lie on 16 bytes
template <typename TQ, bool SILU>
__global__ __launch_bounds__(kLwThreads) void lightning_walk_prep_kernel(const LinearStep a, int at_most, const float* __restrict__ decay, int dp,
                                                                         int vec) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int KS = dp + 4;
  float* Qs = lds;                               // [32][KS]
  float* Ks = Qs + kLwChunk * KS;                // [32][KS]
  float* pw = Ks + kLwChunk * KS;                // [33] powers of the decay, by repeated multiplication
  int seq = 0, tok0 = 0, before = 0;
  const int cn = find_run_piece(a.q_start, a.num_seqs, at_most, kLwChunk, blockIdx.x, &seq, &tok0, &before);
  if (cn <= 0) return;                           // the whole workgroup
  const int h = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int64_t row0 = a.q_start[seq] + tok0;
  float* rec = a.workspace + ((int64_t)blockIdx.x * a.heads + h) * lw_record(dp);
  float4* Qg = reinterpret_cast<float4*>(rec);
  float4* Kt = reinterpret_cast<float4*>(rec + 32 * (int64_t)dp);
  float* keep = rec + 64 * (int64_t)dp;
  float* A = rec + 65 * (int64_t)dp;
  if (tid == 0) {
    const double lam = decay[h];                 // 64 bits: a chunk's 32 roundings would add up over a long run
    double p = 1.0;
    for (int e = 0; e <= kLwChunk; ++e) {
      pw[e] = (float)p;
      p *= lam;
    }
  }
  for (int e = tid; e < kLwChunk * dp / 8; e += kLwThreads) {
    const int r = e / (dp / 8), c = (e - r * (dp / 8)) * 8;
    const int64_t at = (row0 + r) * a.qk_stride + (int64_t)h * a.dim;
    float q[8], k[8];
    lw_load8<TQ>(q, a.q, at, c, a.dim, r < cn, vec != 0);
    lw_load8<TQ>(k, a.k, at, c, a.dim, r < cn, vec != 0);
    if (SILU) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {              // silu(0) = 0
        q[j] = fast_siluf_(q[j]);
        k[j] = fast_siluf_(k[j]);
      }
    }
    lw_put8(Qs + r * KS + c, q);
    lw_put8(Ks + r * KS + c, k);
  }
  __syncthreads();
  for (int e = tid; e < 8 * dp; e += kLwThreads) {
    const int r = (e >> 6 & 1) * 16 + (e & 15), c = (e >> 7) * 16 + (e >> 4 & 3) * 4;
    const float4 q = *reinterpret_cast<const float4*>(Qs + r * KS + c);
    const float f = pw[r + 1];
    Qg[lw_q_quad(r, c)] = make_float4(q.x * f, q.y * f, q.z * f, q.w * f);
  }
  for (int e = tid; e < 8 * dp; e += kLwThreads) {
    const int c = (e >> 7) * 16 + (e & 15), t = (e >> 4 & 7) * 4;
    float k[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) k[j] = Ks[(t + j) * KS + c] * pw[max(cn - 1 - t - j, 0)];    // rows beyond the chunk are zeros
    Kt[lw_k_quad(t, c)] = make_float4(k[0], k[1], k[2], k[3]);
  }
  for (int c = tid; c < dp; c += kLwThreads) keep[c] = pw[cn];
  if (wave < 3) {
    const int li = lane & 15, gq = lane >> 4, bi = wave == 0 ? 0 : 1, bj = wave == 1 ? 1 : 0;
    const f32x4 w = lw_block(Qs + bi * 16 * KS, Ks + bj * 16 * KS, KS, dp);
    f32x4 a;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * bi + li, j = 16 * bj + 4 * gq + r;
      a[r] = j <= i ? w[r] * pw[max(i - j, 0)] : 0.0f;
    }
    reinterpret_cast<f32x4*>(A)[(bi + bj) * 64 + lane] = a;
  }
}

// What a chunk brings to a wave of the state's ...
struct LwState {
  f32x4 kt[2][2];                                // [16 coordinates][16 tokens]: coordinate l % 16, tokens 4 (l / 16) ..
  f32x4 keep[2];                                 // coordinates 16 i + 4 (l / 16) ..
};
// ... and to one of the outputs', which also has some of the tasks kLwValues: the values, kLwTile << i: the outputs of token tile i
template <typename TV>
struct LwOutputs {
  f32x4 q[2][2];                                 // [16 tokens][16 coordinates]: token l % 16, coordinates 4 (l / 16) ..
  f32x4 a[3];
  typename Conv<TV>::store_t v[2][4];            // tokens 16 i + 4 (l / 16) + r of this lane's channel
};
constexpr int kLwValues = 1, kLwTile = 2;
// a quad at `base`, the same for all lanes, and an offset in bytes
__device__ __forceinline__ f32x4 lw_quad(const float* base, uint32_t offset) {
  return *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(base) + offset);
}
__device__ __forceinline__ f32x4 lw_mfma(const f32x4& a, const f32x4& b, f32x4 c) {
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
  return c;
}
// The barrier of a chunk.  The state's waves and the outputs' meet at it from loops of their own, as often: once a chunk and once
// behind the last one.
__device__ __forceinline__ void lw_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
// Waits for all loads.  In front of a loop whose loads are asked for ahead: the compiler counts what is in flight at the loop's head
// as the least of both ways in, and would wait for newer loads than it needs on every turn.
__device__ __forceinline__ void lw_loads_done() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// A walk's pieces of runs: whole ones, or segments.  A segment's place in the scratch: [state: 16-channel block | 32 coordinates |
// tile | lane], the accumulators' layout, and the products of its decays.
struct LwPieces {
  int at_most, segment;                          // 0: whole runs
  int64_t items;
  float *states, *decays;                        // [items][heads][16 vblocks dp], [items][heads][dp]
};

// The segments' own ends, side by side: a run's first segment from the true state, the others from nothing; the last one is left
// out, and its place takes a copy of the true state, which the walk of the first segment starts from (the state's own place is
// written by the last segment's, at a time of its own).
template <typename TV, bool SILU, int NDB>
__global__ __launch_bounds__(64 * NDB) void linear_segment_kernel(const LinearStep a, const LwPieces pc) {
  constexpr int DP = NDB * 32;
  const int vblocks = (a.vdim + kLwChannels - 1) / kLwChannels;
  const int unit = (blockIdx.x >> 3) / vblocks * 8 + (blockIdx.x & 7), vb = (blockIdx.x >> 3) % vblocks;
  const int item = unit / a.heads, h = unit - item * a.heads;
  int seq = 0, tok0 = 0, before = 0;
  const int n = item < pc.items ? find_run_piece(a.q_start, a.num_seqs, pc.at_most, pc.segment, item, &seq, &tok0, &before) : 0;
  if (n <= 0) return;                            // the whole workgroup
  const int run = a.q_start[seq + 1] - a.q_start[seq], behind = (run - tok0 - 1) / pc.segment;      // segments behind this one
  if (behind == 0) return;                       // (n is a whole segment otherwise)
  const int b = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, gq = lane >> 4;
  const int64_t row0 = (int64_t)a.q_start[seq] + tok0, chunk0 = before + tok0 / kLwChunk;
  const int vc = min(vb * kLwChannels + li, a.vdim - 1);     // (lanes beyond the last channel do its work over again, as in the walk)
  auto place = [&](int64_t it) {
    return reinterpret_cast<f32x4*>(pc.states + ((it * a.heads + h) * vblocks + vb) * (kLwChannels * DP)) + b * 128 + lane;
  };
  f32x4 S[2], D[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    S[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    D[i] = f32x4{1.0f, 1.0f, 1.0f, 1.0f};
    if (tok0 == 0) {
      const float* sp = a.state + ((int64_t)a.state_slot[seq] * a.heads + h) * (int64_t)a.dim * a.vdim;
      const bool fresh = a.ctx_len[seq] == 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = 32 * b + 16 * i + 4 * gq + r;
        S[i][r] = (!fresh && c < a.dim) ? sp[(int64_t)c * a.vdim + vc] : 0.0f;
      }
      place(item + behind)[64 * i] = S[i];
    }
  }
  const typename Conv<TV>::store_t* vsrc = static_cast<const typename Conv<TV>::store_t*>(a.v) + row0 * a.v_stride +
                                           (int64_t)h * a.vdim + vc;
  struct Ops {
    f32x4 kt[2][2], keep[2];
    typename Conv<TV>::store_t v[2][4];
  };
  const int chunks = pc.segment / kLwChunk;
  auto fetch = [&](Ops& x, int ci) {
    const float* rec = a.workspace + ((chunk0 + ci) * a.heads + h) * lw_record(DP);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        x.kt[i][j] = lw_quad(rec + 32 * DP + b * 1024, lane * 16 + (2 * i + j) * 1024);
      x.keep[i] = *reinterpret_cast<const f32x4*>(rec + 64 * DP + 32 * b + 16 * i + 4 * gq);
#pragma unroll
      for (int r = 0; r < 4; ++r) x.v[i][r] = vsrc[(ci * kLwChunk + 16 * i + 4 * gq + r) * a.v_stride];
    }
  };
  auto chunk = [&](const Ops& x) {
    f32x4 v[2], add[2] = {};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float y = Conv<TV>::to_float(x.v[i][r]);
        v[i][r] = SILU ? fast_siluf_(y) : y;
      }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i) add[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kt[i][j][r], v[j][r], add[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      S[i] = S[i] * x.keep[i] + add[i];
      D[i] *= x.keep[i];
    }
  };
  Ops x0, x1;
  fetch(x0, 0);
#pragma unroll 1
  for (int ci = 0; ci < chunks; ci += 2) {
    fetch(x1, min(ci + 1, chunks - 1));
    __builtin_amdgcn_sched_barrier(0);
    chunk(x0);
    if (ci + 1 >= chunks) break;
    fetch(x0, min(ci + 2, chunks - 1));
    __builtin_amdgcn_sched_barrier(0);
    chunk(x1);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    place(item)[64 * i] = S[i];
    if (vb == 0 && li == 0)
      *reinterpret_cast<f32x4*>(pc.decays + ((int64_t)item * a.heads + h) * DP + 32 * b + 16 * i + 4 * gq) = D[i];
  }
}

// Piece unit / heads of head unit % heads, 16 value channels of it; false when there is no such piece (and none behind it).
// (No barrier is needed between two calls: what the readers of the last chunk may still read is written behind the next call's first.)
template <typename TV, bool SILU, int NDB>
__device__ __forceinline__ bool linear_walk_piece(const LinearStep& a, const LwPieces& pc, int unit, int vb, int vblocks, int tid) {
  __shared__ f32x4 states[2][NDB][2][64];        // [chunk parity][32 coordinates][16 coordinates][lane]: S_0
  __shared__ f32x4 queried[2][NDB][2][64];       // [chunk parity][wave][token tile][lane]: shares of Q~ S_0
  __shared__ f32x4 values[2][2][64];             // [chunk parity][token tile][lane]: V
  constexpr int DP = NDB * 32, kAhead = NDB <= 4 ? 2 : 1;
  const int item = unit / a.heads, h = unit - item * a.heads;
  int seq = 0, tok0 = 0, before = 0;
  const int n = item < pc.items ? find_run_piece(a.q_start, a.num_seqs, pc.at_most, pc.segment > 0 ? pc.segment : 1 << 30, item, &seq,
                                                &tok0, &before)
                                : 0;
  if (n <= 0) return false;                      // the whole workgroup
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), b = wave % NDB;
  const int lane = tid & 63, li = lane & 15, gq = lane >> 4;
  const int64_t row0 = (int64_t)a.q_start[seq] + tok0, chunk0 = before + tok0 / kLwChunk;
  // This lane's value channel; lanes beyond the last one do its work over again, which spares the stores a condition.
  const int vc = min(vb * kLwChannels + li, a.vdim - 1);
  const int chunks = (n + kLwChunk - 1) / kLwChunk;
  // Where the next chunk's operands lie.  A load of 64 quads is then a base in scalar registers, a lane's 16 bytes and a constant.
  const int64_t rec_step = a.heads * lw_record(DP);
  const float* rec_at = a.workspace + (chunk0 * a.heads + h) * lw_record(DP);
  const uint32_t lane16 = lane * 16;
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  int fetched = 0;
  auto next_chunk = [&]() {                      // (behind the last chunk there is only the last chunk once more)
    rec_at += ++fetched < chunks ? rec_step : 0;
  };
  // The schedules are written out: a load, or a few vector instructions, behind each product, which takes the matrix core 32 cycles.
  if (wave < NDB) {
    // ------------------------------------------------------------------------------------------------------------ the state
    const int run = a.q_start[seq + 1] - a.q_start[seq];
    float* sp = a.state + ((int64_t)a.state_slot[seq] * a.heads + h) * (int64_t)a.dim * a.vdim;
    f32x4 S[2];
    const bool fresh = a.ctx_len[seq] == 0, last = tok0 + n >= run;
    if (pc.segment > 0 && !(tok0 == 0 && last)) {  // a segment: the true state behind the ones in front of it
      const int index = tok0 / pc.segment, first = item - index, end = first + (run - 1) / pc.segment;
      auto place = [&](int64_t it) {
        return reinterpret_cast<const f32x4*>(pc.states + ((it * a.heads + h) * vblocks + vb) * (kLwChannels * DP)) + b * 128 + lane;
      };
#pragma unroll
      for (int i = 0; i < 2; ++i) S[i] = place(index == 0 ? end : first)[64 * i];
#pragma unroll 4
      for (int it = first + 1; it < item; ++it) {
        const float* d = pc.decays + ((int64_t)it * a.heads + h) * DP + 32 * b + 4 * gq;
#pragma unroll
        for (int i = 0; i < 2; ++i) S[i] = S[i] * *reinterpret_cast<const f32x4*>(d + 16 * i) + place(it)[64 * i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = 32 * b + 16 * i + 4 * gq + r;
          S[i][r] = (!fresh && c < a.dim) ? sp[(int64_t)c * a.vdim + vc] : 0.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) states[0][b][i][lane] = S[i];
    auto fetch = [&](LwState& x, int part) {     // one of the 5 portions of a chunk's loads
      if (part < 4) x.kt[part >> 1][part & 1] = lw_quad(rec_at + 32 * DP + b * 1024, lane16 + part * 1024);
      if (part == 4) {
#pragma unroll
        for (int i = 0; i < 2; ++i) x.keep[i] = lw_quad(rec_at + 64 * DP + 32 * b + 16 * i, gq * 16);
        next_chunk();
      }
    };
    auto chunk = [&](const LwState& x, LwState& next, int buf, bool more) {
      lw_barrier();                              // (two buffers: nobody is more than a chunk ahead of a reader)
      f32x4 v[2], add[2] = {zero, zero};         // summed by itself: the state is rounded once a chunk, not once a token
#pragma unroll
      for (int i = 0; i < 2; ++i) v[i] = values[buf][i][lane];
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const int j = s >> 3, r = (s >> 1) & 3, i = s & 1;
        add[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kt[i][j][r], v[j][r], add[i], 0, 0, 0);
        if (more && s % 3 == 1) fetch(next, s / 3);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        S[i] = S[i] * x.keep[i] + add[i];
        states[buf ^ 1][b][i][lane] = S[i];
      }
    };
    LwState x[kAhead + 1];
#pragma unroll
    for (int s = 0; s < kAhead; ++s)
#pragma unroll
      for (int p = 0; p < 5; ++p) fetch(x[s], p);
    lw_loads_done();
    int ci = 0;
#pragma unroll 1
    for (; ci + kAhead < chunks; ci += kAhead + 1)
#pragma unroll
      for (int s = 0; s <= kAhead; ++s) chunk(x[s], x[(s + kAhead) % (kAhead + 1)], (ci + s) & 1, true);
#pragma unroll
    for (int s = 0; s < kAhead; ++s)
      if (ci + s < chunks) chunk(x[s], x[kAhead], (ci + s) & 1, false);
    lw_barrier();
    if (last) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = 32 * b + 16 * i + 4 * gq + r;
          if (c < a.dim) sp[(int64_t)c * a.vdim + vc] = S[i][r];
        }
    }
    return true;
  }
  // ------------------------------------------------------------------------------------------------------------ the outputs
  // O = A V + Q~ S_0: the shares of Q~ S_0 meet behind the next chunk's barrier.  The values are widened a chunk ahead of the state.
  using store_t = typename Conv<TV>::store_t;
  const int64_t out_row = (int64_t)a.heads * a.vdim;
  auto outputs = [&](auto tasks) {
    constexpr int kTasks = decltype(tasks)::value;
    const store_t* const v0 = static_cast<const store_t*>(a.v) + row0 * a.v_stride + (int64_t)h * a.vdim + vc;
    const store_t* v_at = v0 + 4 * gq * a.v_stride;          // of the chunk whose values are fetched next
    int v_tok = 4 * gq;                          // this lane's first token of it
    int w_tok = 4 * gq;                          // ... and of the chunk whose values are widened next
    auto fetch = [&](LwOutputs<TV>& x, int part) {           // one of the 5 portions of a chunk's loads
      if (part < 4) x.q[part >> 1][part & 1] = lw_quad(rec_at + b * 1024, lane16 + part * 1024);
      if (part == 0 && (kTasks & kLwTile)) x.a[0] = lw_quad(rec_at + 65 * DP, lane16);
      if ((part == 1 || part == 2) && (kTasks & 2 * kLwTile)) x.a[part] = lw_quad(rec_at + 65 * DP + part * 256, lane16);
      if (part == 4) next_chunk();
    };
    auto fetch_values = [&](LwOutputs<TV>& x, int part) {    // one of 4 portions, 3 moves on
      if ((kTasks & kLwValues) == 0) return;
#pragma unroll
      for (int r = 2 * (part & 1); r < 2 * (part & 1) + 2; ++r) {
        const int t = 16 * (part >> 1) + r;
        x.v[part >> 1][r] = *(v_tok + t < n ? v_at + t * a.v_stride : v0);
      }
      if (part == 3) {
        v_tok += kLwChunk;
        v_at += kLwChunk * a.v_stride;
      }
    };
    auto widen = [&](const LwOutputs<TV>& x, int buf) {
      if ((kTasks & kLwValues) == 0) return;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) {            // (the padding read some other token's value)
          const float y = w_tok + 16 * i + r < n ? Conv<TV>::to_float(x.v[i][r]) : 0.0f;
          v[r] = SILU ? fast_siluf_(y) : y;
        }
        values[buf][i][lane] = v;
      }
      w_tok += kLwChunk;
    };
    f32x4 av[2] = {zero, zero};
    int o_tok = 0;                               // the first token of the chunk that is finished next
    float* o_at = a.out + ((row0 + 4 * gq) * a.heads + h) * (int64_t)a.vdim + vc;
    // Stores under a condition would have the compiler wait for loads as if there had been none, and so for the newest ones.
    // whole: all of the chunk's tokens are there.  In front of the first chunk: what is stored there is overwritten.
    auto finish = [&](const f32x4 (&q)[2], bool whole, bool first) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if ((kTasks & (kLwTile << i)) == 0) continue;
        const f32x4 o = av[i] + q[i];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (whole || o_tok + 4 * gq + 16 * i + r < n) o_at[(16 * i + r) * out_row] = o[r];
      }
      o_tok += first ? 0 : kLwChunk;
      o_at += first ? 0 : kLwChunk * out_row;
    };
    auto collect = [&](f32x4 (&q)[2], int buf) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if ((kTasks & (kLwTile << i)) == 0) continue;
        f32x4 part[NDB];
#pragma unroll
        for (int w = 0; w < NDB; ++w) part[w] = queried[buf][w][i][lane];
        q[i] = part[0];
#pragma unroll
        for (int w = 1; w < NDB; ++w) q[i] += part[w];
      }
    };
    auto chunk = [&](const LwOutputs<TV>& x, LwOutputs<TV>& next, int ci, bool more) {
      const int buf = ci & 1;
      lw_barrier();
      f32x4 S[2], qs[2] = {zero, zero}, q[2], v[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) S[i] = states[buf][b][i][lane];
      if (kTasks & (3 * kLwTile)) {
        if (more || ci > 0) collect(q, buf ^ 1);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (i == 0 || (kTasks & 2 * kLwTile)) v[i] = values[buf][i][lane];
      }
      if (more || ci + 1 < chunks) widen(x, buf ^ 1);
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const int j = s >> 3, r = (s >> 1) & 3, i = s & 1;
        qs[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[i][j][r], S[j][r], qs[i], 0, 0, 0);
        if (more && s % 3 == 1) fetch(next, s / 3);
        if (more && s % 4 == 2) fetch_values(next, s / 4);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) queried[buf][b][i][lane] = qs[i];
      if (more || ci > 0) finish(q, true, ci == 0);
      if (kTasks & kLwTile) av[0] = lw_mfma(x.a[0], v[0], zero);
      if (kTasks & 2 * kLwTile) av[1] = lw_mfma(x.a[2], v[1], lw_mfma(x.a[1], v[0], zero));
    };
    // stage s holds chunk s's operands and the values of chunk s + 1; those of the first chunk are used at once
    LwOutputs<TV> x[kAhead + 1];
    if (kTasks & kLwValues) {
#pragma unroll
      for (int p = 0; p < 4; ++p) fetch_values(x[0], p);
      widen(x[0], 0);
    }
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
#pragma unroll
      for (int p = 0; p < 5; ++p) fetch(x[s], p);
#pragma unroll
      for (int p = 0; p < 4; ++p) fetch_values(x[s], p);
    }
    lw_loads_done();
    int ci = 0;
#pragma unroll 1
    for (; ci + kAhead < chunks; ci += kAhead + 1)
#pragma unroll
      for (int s = 0; s <= kAhead; ++s) chunk(x[s], x[(s + kAhead) % (kAhead + 1)], ci + s, true);
#pragma unroll
    for (int s = 0; s < kAhead; ++s)
      if (ci + s < chunks) chunk(x[s], x[kAhead], ci + s, false);
    lw_barrier();
    f32x4 q[2];
    collect(q, (chunks - 1) & 1);
    finish(q, false, false);
  };
  if constexpr (NDB == 1) {
    outputs(std::integral_constant<int, kLwValues | 3 * kLwTile>{});
  } else {
    if (b == 0) outputs(std::integral_constant<int, NDB == 2 ? kLwValues | kLwTile : kLwValues>{});
    if (b == 1) outputs(std::integral_constant<int, 2 * kLwTile>{});
    if constexpr (NDB > 2) {
      if (b == 2) outputs(std::integral_constant<int, kLwTile>{});
      if constexpr (NDB > 3) {
        if (b > 2) outputs(std::integral_constant<int, 0>{});
      }
    }
  }
  return true;
}

// MANY: a workgroup goes on to further pieces, as far as there are any (linear_plan.h says when).
template <typename TV, bool SILU, int NDB, bool MANY>
__global__ __launch_bounds__(128 * NDB, 2) void linear_walk_kernel(const LinearStep a, const LwPieces pc) {
  const int vblocks = (a.vdim + kLwChannels - 1) / kLwChannels;
  const int first = (blockIdx.x >> 3) / vblocks * 8 + (blockIdx.x & 7), vb = (blockIdx.x >> 3) % vblocks;
  if constexpr (!MANY) {
    linear_walk_piece<TV, SILU, NDB>(a, pc, first, vb, vblocks, threadIdx.x);
  } else {
#pragma unroll 1
    for (int unit = first;; unit += gridDim.x / vblocks) {
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));              // nothing of a piece's is worked out in front of the loop, and kept
      if (!linear_walk_piece<TV, SILU, NDB>(a, pc, unit, vb, vblocks, tid)) return;
    }
  }
}

template <typename K>
inline hipError_t lw_allow_lds(K kernel, size_t bytes) {
  if (bytes <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

template <typename TV, bool SILU>
int launch_walk(const LinearStep& a, const LinearWalkPlan& plan, hipStream_t stream) {
  const int64_t dp = (a.dim + 31) / 32 * 32, vblocks = (a.vdim + kLwChannels - 1) / kLwChannels;
  const int64_t groups = linear_walk_groups(plan, a.heads, a.vdim), walkers = linear_walkers(plan, a.heads, a.dim, a.vdim);
  SW_CHECK_ARG(groups < (1ll << 31), "linear attention: too many sequences and heads");
  LwPieces pc{plan.at_most, plan.segment, plan.items, nullptr, nullptr};
  if (plan.segment > 0) {
    pc.states = a.workspace + plan.chunks * a.heads * lw_record((int)dp);
    pc.decays = pc.states + plan.items * a.heads * kLwChannels * vblocks * dp;
  }
#define SWM_LW_CASE(N)                                                                                                 \
  case N:                                                                                                              \
    if (plan.segment > 0) {                                                                                            \
      hipLaunchKernelGGL((linear_segment_kernel<TV, SILU, N>), dim3((unsigned)groups), dim3(64 * N), 0, stream, a, pc); \
      SW_CHECK_LAUNCH();                                                                                               \
    }                                                                                                                  \
    if (walkers < groups)                                                                                              \
      hipLaunchKernelGGL((linear_walk_kernel<TV, SILU, N, true>), dim3((unsigned)walkers), dim3(128 * N), 0, stream, a, pc); \
    else                                                                                                               \
      hipLaunchKernelGGL((linear_walk_kernel<TV, SILU, N, false>), dim3((unsigned)groups), dim3(128 * N), 0, stream, a, pc); \
    break;
  switch ((a.dim + 31) / 32) {
    SWM_LW_CASE(1)
    SWM_LW_CASE(2)
    SWM_LW_CASE(3)
    SWM_LW_CASE(4)
    SWM_LW_CASE(5)
    SWM_LW_CASE(6)
    SWM_LW_CASE(7)
    SWM_LW_CASE(8)
  }
#undef SWM_LW_CASE
  SW_CHECK_LAUNCH();
  return SW_OK;
}

inline bool lw_aligned(const LinearStep& a, int dtype) {
  const int per16 = dtype == SW_F32 ? 4 : 8;
  return a.dim % 8 == 0 && a.qk_stride % per16 == 0 &&
         (reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k)) % 16 == 0;
}

int gla_walk(const LinearStep& a, const LinearWalkPlan& plan, const void* decay_pre, int64_t decay_stride, const float* decay_bias, float inv_tau, float q_scale,
             int act_dtype, hipStream_t stream) {
  const int dp = (a.dim + 31) / 32 * 32;
  const size_t bytes = sizeof(float) * (80 * (size_t)(dp + 4) + 3 * dp + 4);
  const dim3 grid((unsigned)plan.chunks, (unsigned)a.heads);       // an upper bound of the chunks
  SWM_DISPATCH_ACT(act_dtype, SW_CHECK_HIP(lw_allow_lds(gla_walk_prep_kernel<T>, bytes));
                   hipLaunchKernelGGL(gla_walk_prep_kernel<T>, grid, dim3(kLwThreads), bytes, stream, a, plan.at_most, decay_pre, decay_stride,
                                      decay_bias, inv_tau, q_scale, dp);
                   SW_CHECK_LAUNCH();
                   return (launch_walk<T, false>(a, plan, stream)););
}

int lightning_walk(const LinearStep& a, const LinearWalkPlan& plan, const float* decay, bool silu, int q_dtype, int v_dtype, hipStream_t stream) {
  const int dp = (a.dim + 31) / 32 * 32;
  const size_t bytes = sizeof(float) * (64 * (size_t)(dp + 4) + kLwChunk + 4);
  const int vec = lw_aligned(a, q_dtype);
  const dim3 grid((unsigned)plan.chunks, (unsigned)a.heads);       // an upper bound of the chunks
  if (silu) {                                    // one projection: q, k and v of one type
    SWM_DISPATCH_ACT(q_dtype, SW_CHECK_HIP(lw_allow_lds(lightning_walk_prep_kernel<T, true>, bytes));
                     hipLaunchKernelGGL((lightning_walk_prep_kernel<T, true>), grid, dim3(kLwThreads), bytes, stream, a, plan.at_most, decay, dp, vec);
                     SW_CHECK_LAUNCH();
                     return (launch_walk<T, true>(a, plan, stream)););
  }
  SW_CHECK_HIP(lw_allow_lds(lightning_walk_prep_kernel<float, false>, bytes));
  hipLaunchKernelGGL((lightning_walk_prep_kernel<float, false>), grid, dim3(kLwThreads), bytes, stream, a, plan.at_most, decay, dp, vec);
  SW_CHECK_LAUNCH();
  SWM_DISPATCH_ACT(v_dtype, return (launch_walk<T, false>(a, plan, stream)););
}

}  // namespace swm
