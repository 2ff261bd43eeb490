// The delta rule with a gate and ONE decay per head in chunks of 32 tokens, for steps that bring long runs:
//     S <- g_t S;  u_t = beta_t (v_t - S^T k_t);  S <- S + k_t u_t^T;  o_t = S^T q_t         (S [dim, vdim], fp32)
// With L_t = log g_1 + ... + log g_t inside a chunk (<= 0, so every ratio e^(L_t - L_s), s <= t, is at most 1) and S_0
// the state at the chunk's start, the chunk's u_t solve (I + A) U = W,  W = diag(beta) (V - diag(e^L) K S_0), with the strict
// lower triangle A[t, s] = beta_t e^(L_t - L_s) (k_t . k_s).  T = (I + A)^-1 does not depend on the state, so
//   a PROLOGUE, parallel over (chunk, key head, two of its value heads), makes unit q and k and for each value head beta, L,
//   P[t, s] = e^(L_t - L_s) (q_t . k_s) (s <= t), T and -T diag(beta e^L) K, the W of the walk;
//   the WALK goes through a sequence's chunks with   U = T diag(beta) V + W S_0,   O = diag(e^L) Q S_0 + P U,
//   S_n = e^(L_n) S_0 + K^T diag(e^(L_n - L)) U,  fp32 products on the matrix cores, which is the recurrence with its sums
//   reordered.
//
// What bounds the walk is its chain: chunk after chunk, product after product, so whatever does not depend on the state is kept
// out of it.  A workgroup owns (sequence, head, 16 value channels) and has two waves per 32 key coordinates: one of the CHAIN, which
// keeps the state's coordinates 32 b .. 32 b + 31 in the accumulators of v_mfma_f32_16x16x4_f32 (lane l: channel l % 16; element r
// of tile i: coordinate 32 b + 16 i + 4 (l / 16) + r), which is also how the B operand of the next product wants them, and one of the
// OUTPUTS, which takes the state from LDS and runs beside the chain's next chunk (Q S_0, P U, T diag(beta) V a chunk ahead, all
// stores).  The waves' shares of W S_0 meet in LDS behind the one barrier of a chunk.  What a chunk brings comes straight from
// memory into registers, two chunks ahead, from a workspace that has it in the lanes' order, so that every load is a whole
// kilobyte.  Workgroups that read the same chunks (the channels of a head) have numbers 8 apart: one XCD, one L2.
// Measured, two prompts of 4324 tokens together, 16 heads on 8 of 128: prologue 69 us and walk 233 us with W = T (beta V - beta e^L
// K S_0) in the chain, operands in rows and one wave per 32 coordinates for all products; 31 and 118 us here.  Of the walk's 1.5 us a
// chunk the products are 0.8 (60 of 32 cycles on the busiest SIMD), products, exchange and stores without the loads 1.0; 57 KB
// of operands a chunk and compute unit through the L1 are the rest.  U_0 = T diag(beta) V made by the prologue as well: 43 and 117
// (the prologue is at the memory's rate then); Q and P multiplied out against the state the same way, O = Q' S_0 + O_0: 55 and 106.
// L is summed in 64 bits: its differences are what counts, and where decays are strong 32 bits leave the end states an error of
// 0.5 - 1.3e-6 (1.2 - 1.5e-7 here).
// Rows of a last, shorter chunk are padded with beta = 0, k = 0, g = 1: they change nothing and are not stored.
#include "delta_step.h"
#include "mixers_common.cuh"

#include <algorithm>
#include <type_traits>

namespace swm {

using f32x4 = __attribute__((ext_vector_type(4))) float;
constexpr int kDcChunk = 32;
constexpr int kDcPrepThreads = 256;
constexpr int kDcPrepHeads = 2;          // value heads of a prologue's workgroup
constexpr int kDcShort = 16;             // tokens of a sequence that goes the decode kernel's way in a mixed step
constexpr int kDcChannels = 16;          // value channels of a walk's workgroup

// The workspace holds the operands of the walk's products in the order in which its lanes read them: FRAGMENTS of 64 quads, one a
// lane, of a 16 x 16 tile.  Floats of one (chunk, key head): K^T by [32 coordinates][16 coordinates][16 tokens] | Q by
// [32 coordinates][16 tokens][16 coordinates] ...
__host__ __device__ constexpr int64_t dc_keys_floats(int dp) { return 64 * (int64_t)dp; }
// ... and of one (chunk, value head): W as Q | tiles (0, 0), (1, 0), (1, 1) of T diag(beta) | of P | e^L | e^(L_n - L) | e^(L_n), 16 times
constexpr int kDcT = 0, kDcP = 768, kDcEl = 1536, kDcTail = 1568, kDcKeep = 1600;             // behind W
__host__ __device__ constexpr int64_t dc_record_floats(int dp) { return 32 * (int64_t)dp + 1616; }

// the prologue's LDS: keys and queries [32][dp + 4]; in their place, per value head, 5 tiles, 2 vectors and one of 64 bits
constexpr int kDcHeadQuads = 5 * 64 + 4 * 8;
__host__ __device__ constexpr int dc_prep_keys_floats(int dp) {
  return 2 * kDcChunk * (dp + 4) > 4 * kDcPrepHeads * kDcHeadQuads ? 2 * kDcChunk * (dp + 4) : 4 * kDcPrepHeads * kDcHeadQuads;
}

__device__ __forceinline__ f32x4 dc_mfma(const f32x4& a, const f32x4& b, f32x4 c) {
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
  return c;
}
// what a wave wrote to LDS is what its lanes read next
__device__ __forceinline__ void dc_wave_sync() {
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
}

// vec: rows of qkv and their parts lie on 16 bytes
template <typename T, int NDB>
__global__ __launch_bounds__(kDcPrepThreads, NDB <= 4 ? 4 : 2) void delta_chunk_prep_kernel(
    float* __restrict__ keys, float* __restrict__ records, const float* __restrict__ qkv, const void* __restrict__ beta_pre,
    int64_t beta_stride, const void* __restrict__ decay_pre, int64_t decay_stride,
    const float* __restrict__ dt_bias, const float* __restrict__ a_log, const int32_t* __restrict__ q_start, int num_seqs,
    int at_most, int heads, int kv_heads, int dim, int vdim, int vec) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int DP = NDB * 32, KS = DP + 4;      // rows on 16 bytes
  float* Kn = lds;                               // [32][KS] unit keys
  float* Qn = Kn + kDcChunk * KS;                // [32][KS] unit queries times dim^-1/2
  f32x4* dots = reinterpret_cast<f32x4*>(lds + dc_prep_keys_floats(DP)); // [K K^T | Q K^T][tile (0, 0) (1, 0) (1, 1)][lane]
  f32x4* heads_lds = reinterpret_cast<f32x4*>(lds);          // later, in their place, per value head: [4 matrices][3 tiles][lane], vectors
  const int group = heads / kv_heads, parts = (group + kDcPrepHeads - 1) / kDcPrepHeads;
  const int g = blockIdx.y / parts, m0 = (blockIdx.y - g * parts) * kDcPrepHeads, nm = min(kDcPrepHeads, group - m0);
  int seq = 0, tok0 = 0, before = 0;
  const int cn = find_run_piece(q_start, num_seqs, at_most, kDcChunk, blockIdx.x, &seq, &tok0, &before);
  if (cn <= 0) return;                           // the whole workgroup
  const int64_t row0 = q_start[seq] + tok0;
  const int64_t row_w = 2 * (int64_t)kv_heads * dim + (int64_t)heads * vdim;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, gq = lane >> 4, l32 = lane & 31;
  // ---- what is read far from its use: a head's decays and betas
  const int h_own = g * group + m0 + min(wave, nm - 1);
  const float beta_raw = ld<T>(beta_pre, (row0 + min(l32, cn - 1)) * beta_stride + h_own);
  const float decay_raw = ld<T>(decay_pre, (row0 + min(l32, cn - 1)) * decay_stride + h_own);
  const float bias = dt_bias[h_own], alog = a_log[h_own];
  // ---- unit queries and keys: 8 lanes a row
  {
    const int r = tid >> 3, p = (tid & 7) * 4;
    const float* src = qkv + (row0 + min(r, cn - 1)) * row_w + (int64_t)g * dim;
    f32x4 q[NDB], k[NDB];
#pragma unroll
    for (int i = 0; i < NDB; ++i) {
      const int c = 32 * i + p;
      if (vec && c < dim) {
        q[i] = *reinterpret_cast<const f32x4*>(src + c);
        k[i] = *reinterpret_cast<const f32x4*>(src + (int64_t)kv_heads * dim + c);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          q[i][j] = c + j < dim ? src[c + j] : 0.0f;
          k[i][j] = c + j < dim ? src[(int64_t)kv_heads * dim + c + j] : 0.0f;
        }
      }
    }
    float qq = 0.0f, kk = 0.0f;
#pragma unroll
    for (int i = 0; i < NDB; ++i) {
      if (r >= cn) q[i] = k[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < 4; ++j) qq += q[i][j] * q[i][j], kk += k[i][j] * k[i][j];
    }
    qq = lanes_sum<8>(qq);
    kk = lanes_sum<8>(kk);
    const float qf = (1.0f / sqrtf((float)dim)) / sqrtf(qq + 1e-6f), kf = 1.0f / sqrtf(kk + 1e-6f);
#pragma unroll
    for (int i = 0; i < NDB; ++i) {
      *reinterpret_cast<f32x4*>(Qn + r * KS + 32 * i + p) = q[i] * qf;
      *reinterpret_cast<f32x4*>(Kn + r * KS + 32 * i + p) = k[i] * kf;
    }
  }
  __syncthreads();
  // ---- K K^T and Q K^T, a tile of each per wave: element r of a lane is row 4 gq + r, column li
  if (wave < 3) {
    const float* kt = Kn + ((wave > 0 ? 16 : 0) + li) * KS + 4 * gq;
    const float* qt = Qn + ((wave > 0 ? 16 : 0) + li) * KS + 4 * gq;
    const float* ks = Kn + ((wave > 1 ? 16 : 0) + li) * KS + 4 * gq;
    f32x4 kk = {0.0f, 0.0f, 0.0f, 0.0f}, qk = kk;
#pragma unroll
    for (int c = 0; c < DP; c += 16) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(kt + c), q = *reinterpret_cast<const f32x4*>(qt + c);
      const f32x4 s = *reinterpret_cast<const f32x4*>(ks + c);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        kk = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], s[r], kk, 0, 0, 0);
        qk = __builtin_amdgcn_mfma_f32_16x16x4f32(q[r], s[r], qk, 0, 0, 0);
      }
    }
    dots[wave * 64 + lane] = kk;
    dots[(3 + wave) * 64 + lane] = qk;
  }
  // ---- the fragments of K^T and Q for the walk; the keys also for the product at the end, a wave's 16 coordinates
  constexpr int kSlices = (2 * NDB + 3) / 4;
  f32x4 k[kSlices][2];
#pragma unroll
  for (int a = 0; a < kSlices; ++a) {
    const int s = min(wave + 4 * a, 2 * NDB - 1);
    f32x4* at = reinterpret_cast<f32x4*>(keys + ((int64_t)blockIdx.x * kv_heads + g) * dc_keys_floats(DP)) + lane;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) k[a][j][r] = Kn[(16 * j + 4 * gq + r) * KS + 16 * s + li];
      if (m0 == 0 && wave + 4 * a < 2 * NDB) {
        at[s * 128 + j * 64] = k[a][j];
        at[8 * DP + (s >> 1) * 256 + j * 128 + (s & 1) * 64] = *reinterpret_cast<const f32x4*>(Qn + (16 * j + li) * KS + 16 * s + 4 * gq);
      }
    }
  }
  __syncthreads();
  // ---- a wave per value head: beta, L, A, P, T = (I + A)^-1; left in LDS: -T diag(beta e^L), as tiles whose quad of lane l is
  //      row l % 16, columns 4 (l / 16) ..
  if (wave < nm) {
    f32x4* F = heads_lds + wave * kDcHeadQuads;
    f32x4 *fa = F, *ft = F + 3 * 64;             // before that: A; the diagonal tiles of T, by columns
    float* vec32 = reinterpret_cast<float*>(F + 5 * 64);     // beta | e^L; running sums of the log decays (64 bits)
    double* Ls = reinterpret_cast<double*>(vec32 + 64);
    float* rec = records + ((int64_t)blockIdx.x * heads + h_own) * dc_record_floats(DP) + 32 * (int64_t)DP;
    float beta = 0.0f;
    double L = 0.0;                              // of token l32, in both halves
    if (l32 < cn) {
      beta = sigmoidf_(beta_raw);
      const float g = -expf(alog) * softplusf_(decay_raw + bias);
      L = g < -200.0f ? -200.0f : g;             // a decay of 0; differences of sums with -inf or -1e30 in them would be of nothing
    }
#pragma unroll
    for (int step = 1; step < 32; step <<= 1) {
      const double o = __shfl_up(L, step, 32);
      if (l32 >= step) L += o;
    }
    const double Ln = __shfl(L, 31, 32);
    if (lane < 32) {
      Ls[l32] = L;
      vec32[l32] = beta;
      vec32[32 + l32] = expf((float)L);
      rec[kDcEl + l32] = vec32[32 + l32];
      rec[kDcTail + l32] = expf((float)(Ln - L));
      if (lane < 16) rec[kDcKeep + lane] = expf((float)Ln);  // (16 times, for the lanes that load it)
    }
    dc_wave_sync();
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const int ti = x > 0 ? 16 : 0, si = x > 1 ? 16 : 0;
      const f32x4 kk = dots[x * 64 + lane], qk = dots[(3 + x) * 64 + lane];
      const double Lc = Ls[si + li];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = ti + 4 * gq + r, s = si + li, at = ((li >> 2) * 16 + 4 * gq + r) * 4 + (li & 3);
        const float ratio = s <= t ? expf((float)(Ls[t] - Lc)) : 0.0f;
        reinterpret_cast<float*>(fa + x * 64)[at] = s < t ? vec32[t] * ratio * kk[r] : 0.0f;
        rec[kDcP + x * 256 + at] = ratio * qk[r];
      }
    }
    dc_wave_sync();
    // the inverses of I + A's diagonal tiles, row by row: T[t, :] = e_t - sum_{s < t} A[t, s] T[s, :], a lane per column
    {
      const f32x4* tile = fa + (gq & 1) * 2 * 64;
      float col[16];
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        float p0 = 0.0f, p1 = 0.0f;
#pragma unroll
        for (int s4 = 0; s4 < (t + 3) / 4; ++s4) {           // (A is zero from the diagonal on)
          const f32x4 x = tile[s4 * 16 + t];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (4 * s4 + j < t) (j & 1 ? p1 : p0) += x[j] * col[4 * s4 + j];
          }
        }
        col[t] = (t == li ? 1.0f : 0.0f) - (p0 + p1);
      }
      if (gq < 2) {
#pragma unroll
        for (int t4 = 0; t4 < 4; ++t4)
          ft[gq * 64 + t4 * 16 + li] = f32x4{col[4 * t4], col[4 * t4 + 1], col[4 * t4 + 2], col[4 * t4 + 3]};
      }
    }
    dc_wave_sync();
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 t[3];                                  // tiles (0, 0), (1, 0), (1, 1): element r is row 4 gq + r, column li
    t[0] = ft[lane];
    t[2] = ft[64 + lane];
    {
      f32x4 row22;                               // row li of the second diagonal tile, columns 4 gq ..
#pragma unroll
      for (int r = 0; r < 4; ++r) row22[r] = -reinterpret_cast<const float*>(ft + 64)[((li >> 2) * 16 + 4 * gq + r) * 4 + (li & 3)];
      t[1] = dc_mfma(row22, dc_mfma(fa[64 + lane], t[0], zero), zero);
    }
    dc_wave_sync();
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const int si = x > 1 ? 16 : 0;
      const float bs = vec32[si + li], el = vec32[32 + si + li];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int at = ((li >> 2) * 16 + 4 * gq + r) * 4 + (li & 3);
        const float tb = t[x][r] * bs;
        rec[kDcT + x * 256 + at] = tb;
        reinterpret_cast<float*>(F + x * 64)[at] = -(tb * el);
      }
    }
  }
  __syncthreads();
  // ---- W (16 coordinates at a time, transposed: element r of a lane is coordinate 4 gq + r of token li)
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int m = 0; m < nm; ++m) {
    const f32x4* F = heads_lds + m * kDcHeadQuads;
    const f32x4 f0 = F[lane], f1 = F[64 + lane], f2 = F[128 + lane];
    f32x4* rec = reinterpret_cast<f32x4*>(records + ((int64_t)blockIdx.x * heads + g * group + m0 + m) * dc_record_floats(DP));
#pragma unroll
    for (int a = 0; a < kSlices; ++a) {
      const int s = wave + 4 * a;
      if (s >= 2 * NDB) break;                   // wave-uniform
      f32x4* at = rec + (s >> 1) * 256 + (s & 1) * 64 + lane;
      at[0] = dc_mfma(k[a][0], f0, zero);
      at[128] = dc_mfma(k[a][1], f2, dc_mfma(k[a][0], f1, zero));
    }
  }
}

// What a chunk brings to a wave of the chain ...
struct DcChain {
  f32x4 w[2][2];                                 // [16 tokens][16 coordinates]: token l % 16, coordinates 4 (l / 16) ..
  f32x4 kt[2][2];                                // [16 coordinates][16 tokens]: coordinate l % 16, tokens 4 (l / 16) ..
  f32x4 tail[2];                                 // e^(L_n - L) of tokens 16 i + 4 (l / 16) ..
  float keep;                                    // e^(L_n)
};
// ... and to one of the outputs', which also has some of the tasks kDcValues << i, kDcTile << i: U_0, the outputs of token tile i
struct DcOutputs {
  f32x4 q[2][2];
  f32x4 t[3], v[2];                              // T diag(beta); values of tokens 16 i + 4 (l / 16) .. and this lane's channel
  f32x4 p[3], el[2];                             // P, e^L
};
constexpr int kDcValues = 1, kDcTile = 4;
// a quad at `base`, the same for all lanes, and an offset in bytes
__device__ __forceinline__ f32x4 dc_quad(const float* base, uint32_t offset) {
  return *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(base) + offset);
}
// The barrier of a chunk.  The chain's waves and the outputs' meet at it from loops of their own, as often: once a chunk and once
// behind the last one.
__device__ __forceinline__ void dc_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Waits for all loads.  In front of a loop whose loads are asked for ahead: the compiler counts what is in flight at the loop's head
// as the least of both ways in, and would wait for newer loads than it needs on every turn.
__device__ __forceinline__ void dc_loads_done() { __builtin_amdgcn_s_waitcnt(0x0f70); }

template <int NDB>
__global__ __launch_bounds__(128 * NDB, 2) void delta_chunk_kernel(
    float* __restrict__ out, const float* __restrict__ keys, const float* __restrict__ records, const float* __restrict__ qkv,
    float* __restrict__ state, const int32_t* __restrict__ q_start, const int32_t* __restrict__ ctx_len,
    const int32_t* __restrict__ state_slot, int num_seqs, int at_most, int64_t runs, int heads, int kv_heads, int dim, int vdim) {
  __shared__ f32x4 shares[2][NDB + 1][2][64];    // [chunk parity][U_0, wave][token tile][lane]: of U
  __shared__ f32x4 queried[2][NDB][2][64];       // ... of Q S_0
  __shared__ f32x4 states[2][NDB][2][64];        // [chunk parity][32 coordinates][16 coordinates][lane]: S_0
  constexpr int DP = NDB * 32, kAhead = NDB <= 4 ? 2 : 1;
  const int vblocks = (vdim + kDcChannels - 1) / kDcChannels;
  const int unit = (blockIdx.x >> 3) / vblocks * 8 + (blockIdx.x & 7), vb = (blockIdx.x >> 3) % vblocks;
  const int run = unit / heads, h = unit - run * heads, g = h / (heads / kv_heads);
  int seq = 0, tok0 = 0, chunk0 = 0;             // chunk0: this sequence's first chunk among the step's
  const int n = run < runs ? find_run_piece(q_start, num_seqs, at_most, 1 << 30, run, &seq, &tok0, &chunk0) : 0;
  if (n <= 0) return;                            // the whole workgroup
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), b = wave % NDB;
  const int lane = threadIdx.x & 63, li = lane & 15, gq = lane >> 4;
  // This lane's value channel; lanes beyond the last one do its work over again, which spares the stores a condition.
  const int vc = min(vb * kDcChannels + li, vdim - 1);
  const int chunks = (n + kDcChunk - 1) / kDcChunk;
  const int64_t row0 = q_start[seq];
  // Where the next chunk's operands lie.  A load of 64 quads is then a base in scalar registers, a lane's 16 bytes and a constant.
  const int64_t rec_step = heads * dc_record_floats(DP), keys_step = kv_heads * dc_keys_floats(DP);
  const float* rec_at = records + ((int64_t)chunk0 * heads + h) * dc_record_floats(DP);
  const float* keys_at = keys + ((int64_t)chunk0 * kv_heads + g) * dc_keys_floats(DP);
  const uint32_t lane16 = lane * 16;
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  int fetched = 0;
  auto next_chunk = [&]() {                      // (behind the last chunk there is only the last chunk once more)
    const bool more = ++fetched < chunks;
    rec_at += more ? rec_step : 0;
    keys_at += more ? keys_step : 0;
  };
  // U, from the waves' shares: the same sum, in the same order, for all who need it
  auto sum_shares = [&](int buf, int i) {
    f32x4 part[NDB + 1];
#pragma unroll
    for (int w = 0; w <= NDB; ++w) part[w] = shares[buf][w][i][lane];
    f32x4 u = part[0];
#pragma unroll
    for (int w = 1; w <= NDB; ++w) u += part[w];
    return u;
  };
  // The schedules are written out: a load, or a few vector instructions, behind each product, which takes the matrix core 32 cycles.
  if (wave < NDB) {
    // ------------------------------------------------------------------------------------------------------------ the chain
    float* sp = state + ((int64_t)state_slot[seq] * heads + h) * (int64_t)dim * vdim;
    f32x4 S[2];
    const bool fresh = ctx_len[seq] == 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = 32 * b + 16 * i + 4 * gq + r;
        S[i][r] = (!fresh && c < dim) ? sp[(int64_t)c * vdim + vc] : 0.0f;
      }
      states[0][b][i][lane] = S[i];
    }
    auto fetch = [&](DcChain& x, int part) {     // one of the 10 portions of a chunk's loads
      const int i = (part >> 1) & 1, j = part & 1;
      if (part < 4) x.w[i][j] = dc_quad(rec_at + b * 1024, lane16 + part * 1024);
      if (part >= 4 && part < 8) x.kt[i][j] = dc_quad(keys_at + b * 1024, lane16 + (part - 4) * 1024);
      if (part == 8) {
        x.tail[0] = dc_quad(rec_at + 32 * DP + kDcTail, gq * 16);
        x.tail[1] = dc_quad(rec_at + 32 * DP + kDcTail + 16, gq * 16);
      }
      if (part == 9) {
        x.keep = (rec_at + 32 * DP + kDcKeep)[li];
        next_chunk();
      }
    };
    auto chunk = [&](const DcChain& x, DcChain& next, int buf, bool more) {
      // ---- this wave's share of U = U_0 + W S_0
      f32x4 u[2] = {zero, zero};
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const int j = s >> 3, r = (s >> 1) & 3, i = s & 1;
        u[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[i][j][r], S[j][r], u[i], 0, 0, 0);
        if (more && s % 3 == 1) fetch(next, s / 3);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) shares[buf][1 + b][i][lane] = u[i];
      f32x4 T[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) T[i] = S[i] * x.keep;
      dc_barrier();                              // (two buffers: nobody is more than a chunk ahead of a reader)
      // ---- S <- e^(L_n) S + K^T diag(e^(L_n - L)) U
#pragma unroll
      for (int i = 0; i < 2; ++i) u[i] = sum_shares(buf, i) * x.tail[i];
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const int j = s >> 3, r = (s >> 1) & 3, i = s & 1;
        T[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kt[i][j][r], u[j][r], T[i], 0, 0, 0);
        if (more && s % 3 == 1) fetch(next, 5 + s / 3);
        if (s >= 8) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        S[i] = T[i];
        states[buf ^ 1][b][i][lane] = S[i];
      }
    };
    DcChain x[kAhead + 1];
#pragma unroll
    for (int a = 0; a < kAhead; ++a)
#pragma unroll
      for (int s = 0; s < 10; ++s) fetch(x[a], s);
    dc_loads_done();
    int ci = 0;
#pragma unroll 1
    for (; ci + kAhead < chunks; ci += kAhead + 1)
#pragma unroll
      for (int a = 0; a <= kAhead; ++a) chunk(x[a], x[(a + kAhead) % (kAhead + 1)], (ci + a) & 1, true);
#pragma unroll
    for (int a = 0; a < kAhead; ++a)
      if (ci + a < chunks) chunk(x[a], x[kAhead], (ci + a) & 1, false);
    dc_barrier();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = 32 * b + 16 * i + 4 * gq + r;
        if (c < dim) sp[(int64_t)c * vdim + vc] = S[i][r];
      }
    return;
  }
  // ------------------------------------------------------------------------------------------------------------ the outputs
  // O = diag(e^L) Q S_0 + P U: the shares of Q S_0 meet behind the next chunk's barrier.  U_0 = T diag(beta) V is made a chunk ahead
  // of the chain.  These waves have the more loads and the stores to ask for, and the chain waits for them at the barrier: they go
  // first (127 us without, 115 with, of the figures at the top).
  __builtin_amdgcn_s_setprio(2);
  const int64_t row_w = 2 * (int64_t)kv_heads * dim + (int64_t)heads * vdim, out_row = (int64_t)heads * vdim;
  auto outputs = [&](auto tasks) {
    constexpr int kTasks = decltype(tasks)::value;
    const float* v_at = qkv + row0 * row_w;      // the first row of the chunk whose values are fetched next
    uint32_t v_offset[2][4];                     // this lane's values of a chunk, in bytes behind its first row
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        v_offset[i][r] = 4 * (uint32_t)((16 * i + 4 * gq + r) * row_w + 2 * (int64_t)kv_heads * dim + (int64_t)h * vdim + vc);
    float* o_at = out + ((row0 + 4 * gq) * heads + h) * (int64_t)vdim + vc;      // of the chunk that is finished next
    auto fetch = [&](DcOutputs& x, int part) {   // one of the 5 portions of a chunk's loads; U_0's operands are the next chunk's
      if (part < 4) x.q[part >> 1][part & 1] = dc_quad(keys_at + 32 * DP + b * 1024, lane16 + part * 1024);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if ((kTasks & (kDcTile << i)) == 0) continue;
        if (part == 0) x.el[i] = dc_quad(rec_at + 32 * DP + kDcEl + 16 * i, gq * 16);
        if (part == 1) x.p[i] = dc_quad(rec_at + 32 * DP + kDcP + i * 256, lane16);
        if (part == 2 && i == 1) x.p[2] = dc_quad(rec_at + 32 * DP + kDcP + 512, lane16);
      }
      if (part == 4) next_chunk();
    };
    int v_tok = 0;                               // the first token of the chunk whose values are fetched next
    const float* t_at = rec_at + 32 * DP + kDcT; // ... and its T
    auto fetch_values = [&](DcOutputs& x, int part) {        // one of 4 portions, 3 moves on
      if ((kTasks & (3 * kDcValues)) == 0) return;
      if (part < 3 && (kTasks & (part == 0 ? kDcValues : 2 * kDcValues))) x.t[part] = dc_quad(t_at + part * 256, lane16);
      // rows behind the run: the buffer ends there, and they read as zeros
      const auto rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(v_at), 0, (int)(uint32_t)(4 * row_w * max(min(n - v_tok, kDcChunk), 0)),
                                                          0x00020000);
#pragma unroll
      for (int r = 2 * (part & 1); r < 2 * (part & 1) + 2; ++r) {
        if (part > 1 && (kTasks & (2 * kDcValues)) == 0) continue;
        x.v[part >> 1][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows, v_offset[part >> 1][r], 0, 0));
      }
      if (part == 3) {
        v_tok += kDcChunk;
        t_at += v_tok < n ? rec_step : 0;
        v_at += v_tok < n ? kDcChunk * row_w : 0;
      }
    };
    auto make_values = [&](const DcOutputs& x, int buf) {
      if (kTasks & kDcValues) shares[buf][0][0][lane] = dc_mfma(x.t[0], x.v[0], zero);
      if (kTasks & (2 * kDcValues)) shares[buf][0][1][lane] = dc_mfma(x.t[2], x.v[1], dc_mfma(x.t[1], x.v[0], zero));
    };
    f32x4 pu[2] = {zero, zero}, pel[2] = {zero, zero};
    int o_tok = 0;                               // the first token of the chunk that is finished next
    // Stores under a condition would have the compiler wait for loads as if there had been none, and so for the newest ones.
    // whole: all of the chunk's tokens are there.  In front of the first chunk: what is stored there is overwritten.
    auto finish = [&](const f32x4 (&q)[2], bool whole, bool first) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if ((kTasks & (kDcTile << i)) == 0) continue;
        const f32x4 o = q[i] * pel[i] + pu[i];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (whole || o_tok + 4 * gq + 16 * i + r < n) o_at[(16 * i + r) * out_row] = o[r];
      }
      o_tok += first ? 0 : kDcChunk;
      o_at += first ? 0 : kDcChunk * out_row;
    };
    auto collect = [&](f32x4 (&q)[2], int buf) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if ((kTasks & (kDcTile << i)) == 0) continue;
        f32x4 part[NDB];
#pragma unroll
        for (int w = 0; w < NDB; ++w) part[w] = queried[buf][w][i][lane];
        q[i] = part[0];
#pragma unroll
        for (int w = 1; w < NDB; ++w) q[i] += part[w];
      }
    };
    auto chunk = [&](const DcOutputs& x, DcOutputs& next, int ci, bool more) {
      const int buf = ci & 1;
      dc_barrier();
      f32x4 S[2], qs[2] = {zero, zero}, q[2], u[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) S[i] = states[buf][b][i][lane];
      if (kTasks & (kDcTile | 2 * kDcTile)) {
        if (more || ci > 0) collect(q, buf ^ 1);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (i == 0 || (kTasks & 2 * kDcTile)) u[i] = sum_shares(buf, i);
      }
      if (more || ci + 1 < chunks) make_values(x, buf ^ 1);
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
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if ((kTasks & (kDcTile << i)) == 0) continue;
        pel[i] = x.el[i];
        pu[i] = i == 0 ? dc_mfma(x.p[0], u[0], zero) : dc_mfma(x.p[2], u[1], dc_mfma(x.p[1], u[0], zero));
      }
    };
    // stage a holds chunk a's operands and the values of chunk a + 1; those of the first chunk are used at once
    DcOutputs x[kAhead + 1];
    if (kTasks & (3 * kDcValues)) {
#pragma unroll
      for (int s = 0; s < 4; ++s) fetch_values(x[0], s);
      make_values(x[0], 0);
    }
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
#pragma unroll
      for (int s = 0; s < 5; ++s) fetch(x[a], s);
#pragma unroll
      for (int s = 0; s < 4; ++s) fetch_values(x[a], s);
    }
    dc_loads_done();
    int ci = 0;
#pragma unroll 1
    for (; ci + kAhead < chunks; ci += kAhead + 1)
#pragma unroll
      for (int a = 0; a <= kAhead; ++a) chunk(x[a], x[(a + kAhead) % (kAhead + 1)], ci + a, true);
#pragma unroll
    for (int a = 0; a < kAhead; ++a)
      if (ci + a < chunks) chunk(x[a], x[kAhead], ci + a, false);
    dc_barrier();
    f32x4 q[2];
    collect(q, (chunks - 1) & 1);
    finish(q, false, false);
  };
  // the tasks of the output waves: whole products of 4, 8, 4 and 8 instructions
  if constexpr (NDB == 1) {
    outputs(std::integral_constant<int, 3 * kDcValues | 3 * kDcTile>{});
  } else if constexpr (NDB == 2) {
    if (b == 0) outputs(std::integral_constant<int, 2 * kDcValues | kDcTile>{});
    if (b == 1) outputs(std::integral_constant<int, kDcValues | 2 * kDcTile>{});
  } else if constexpr (NDB == 3) {
    if (b == 0) outputs(std::integral_constant<int, 2 * kDcValues>{});
    if (b == 1) outputs(std::integral_constant<int, kDcValues | kDcTile>{});
    if (b == 2) outputs(std::integral_constant<int, 2 * kDcTile>{});
  } else {
    if (b == 0) outputs(std::integral_constant<int, 2 * kDcValues>{});
    if (b == 1) outputs(std::integral_constant<int, 2 * kDcTile>{});
    if (b == 2) outputs(std::integral_constant<int, kDcTile>{});
    if (b == 3) outputs(std::integral_constant<int, kDcValues>{});
    if constexpr (NDB > 4) {
      if (b > 3) outputs(std::integral_constant<int, 0>{});
    }
  }
}

template <typename K>
inline hipError_t dc_allow_lds(K kernel, size_t bytes) {
  if (bytes <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

struct DcStep {
  float* out;
  const float* qkv;
  const void *beta_pre, *decay_pre;
  int64_t beta_stride, decay_stride;
  const float *dt_bias, *a_log;
  float* state;
  const int32_t *q_start, *ctx_len, *state_slot;
  int num_seqs, at_most, heads, kv_heads, dim, vdim, act_dtype;
  int64_t runs, chunks;                 // an upper bound of the chunks: surplus workgroups leave at once
  float* workspace;
};

template <int NDB>
int launch_delta_chunk(const DcStep& a, hipStream_t stream) {
  constexpr int DP = 32 * NDB;
  const int64_t vblocks = (a.vdim + kDcChannels - 1) / kDcChannels;
  const int64_t units = (a.runs * a.heads + 7) / 8 * 8, groups = units * vblocks;
  const int group = a.heads / a.kv_heads, parts = (group + kDcPrepHeads - 1) / kDcPrepHeads;
  SW_CHECK_ARG(groups < (1ll << 31), "gated_delta_chunked: too many sequences and heads");
  float* records = a.workspace;
  float* keys = a.workspace + a.chunks * a.heads * dc_record_floats(DP);
  const int vec = a.dim % 4 == 0 && (2 * (int64_t)a.kv_heads * a.dim + (int64_t)a.heads * a.vdim) % 4 == 0 &&
                  reinterpret_cast<uintptr_t>(a.qkv) % 16 == 0;
  const size_t lds = sizeof(float) * (dc_prep_keys_floats(DP) + 2 * 3 * 256);
  SWM_DISPATCH_ACT(a.act_dtype, SW_CHECK_HIP(dc_allow_lds((delta_chunk_prep_kernel<T, NDB>), lds));
                   hipLaunchKernelGGL((delta_chunk_prep_kernel<T, NDB>), dim3((unsigned)a.chunks, (unsigned)(a.kv_heads * parts)),
                                      dim3(kDcPrepThreads), lds, stream, keys, records, a.qkv, a.beta_pre, a.beta_stride,
                                      a.decay_pre, a.decay_stride, a.dt_bias, a.a_log, a.q_start, a.num_seqs, a.at_most, a.heads,
                                      a.kv_heads, a.dim, a.vdim, vec););
  SW_CHECK_LAUNCH();
  hipLaunchKernelGGL(delta_chunk_kernel<NDB>, dim3((unsigned)groups), dim3(128 * NDB), 0, stream, a.out, keys, records, a.qkv, a.state,
                     a.q_start, a.ctx_len, a.state_slot, a.num_seqs, a.at_most, a.runs, a.heads, a.kv_heads, a.dim, a.vdim);
  SW_CHECK_LAUNCH();
  return SW_OK;
}

}  // namespace swm

extern "C" {

int64_t swm_gated_delta_chunked_workspace_floats(int64_t rows, int num_seqs, int heads, int dim, int vdim) {
  const int dp = (dim + 31) / 32 * 32;
  (void)vdim;
  return (rows / swm::kDcChunk + num_seqs) * heads * (swm::dc_keys_floats(dp) + swm::dc_record_floats(dp));     // as many key heads at most
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
  // The walk has a chunk's places in 32 bits: rows of 128 MiB and more go token by token (whose workspace is the smaller one).
  if (2 * (int64_t)kv_heads * dim + (int64_t)heads * vdim >= 1ll << 25)
    return swm_gated_delta(out, qkv, beta_pre, beta_stride, decay_pre, decay_stride, dt_bias, a_log, state, q_start, ctx_len, state_slot,
                           rows, num_seqs, heads, kv_heads, dim, vdim, workspace, act_dtype, stream);
  // Decoding sequences beside a portion take the decode kernel: their states are read and written in whole rows there, in 64-byte
  // pieces here, and they need no 32-row record.  Not worth the launch where most sequences are long.  (us a call, 12 heads of 96, a
  // portion of 100 tokens beside 11 / 20 / 60 / 250 decoding sequences: 29 / 44 / 87 / 360 all in chunks, 25 / 26 / 35 / 76 so; beside 6
  // 24.1 and 24.7; 2000 tokens beside 11 105.4 and 106.7)
  const bool mixed = num_seqs >= 12 && rows < 128 * (int64_t)num_seqs &&
                     delta_step(out, qkv, beta_pre, beta_stride, decay_pre, decay_stride, 1, dt_bias, a_log, state, q_start, ctx_len,
                                state_slot, num_seqs, heads, kv_heads, dim, vdim, kDcShort, act_dtype, s);
  SW_CHECK_LAUNCH();
  const int at_most = mixed ? kDcShort : 0;
  const int64_t runs = mixed ? std::min<int64_t>(num_seqs, rows / (kDcShort + 1)) : num_seqs;
  if (runs == 0) return SW_OK;
  const DcStep step{out, qkv, beta_pre, decay_pre, beta_stride, decay_stride, dt_bias, a_log, state, q_start, ctx_len, state_slot,
                    num_seqs, at_most, heads, kv_heads, dim, vdim, act_dtype, runs, rows / kDcChunk + runs, workspace};
  switch ((dim + 31) / 32) {
    case 1: return launch_delta_chunk<1>(step, s);
    case 2: return launch_delta_chunk<2>(step, s);
    case 3: return launch_delta_chunk<3>(step, s);
    case 4: return launch_delta_chunk<4>(step, s);
    case 5: return launch_delta_chunk<5>(step, s);
    case 6: return launch_delta_chunk<6>(step, s);
    default: return launch_delta_chunk<7>(step, s);
  }
}

}  // extern "C"
