// Feed-forward experts over rows that were sorted by expert: two grouped "NT" GEMMs (both operands
// contiguous along the reduction), the first with the experts' activation as its epilogue, the second scattering
// its rows back and adding them into an fp32 output.  bf16 runs on the matrix cores (second half of this
// file, where a reduction's size is a multiple of 8); fp32 -- true fp32, no reduced-precision matrix mode -- on LDS-tiled
// vector FMAs.
//
// The host does not know how many rows an expert got (the sort stays on the device), so a grid of tiles has the
// upper bound ceil(pairs / rows of a tile) + experts row tiles and each workgroup finds its (expert, tile) from the
// prefix sums; surplus workgroups leave at once.  Tiles never straddle two experts.
#include "tile_gemm.cuh"

#include <algorithm>
#include <type_traits>

namespace swm {

constexpr int kFfnThreads = kTileThreads;

__device__ __forceinline__ float gelu_erf(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
// activation of an expert's hidden layer: SWM_ACT_GELU (exact gelu), SWM_ACT_RELU2 (the square of relu) or
// SWM_ACT_NONE (the products as they are, for a gated unit that a kernel of its own applies)
__device__ __forceinline__ float expert_act(float z, int activation) {
  if (activation == SWM_ACT_NONE) return z;
  if (activation == SWM_ACT_RELU2) {
    const float r = fmaxf(z, 0.0f);
    return r * r;
  }
  return gelu_erf(z);
}

// A gated hidden layer with limits, fused into the up-projection: an expert's matrix then holds, per run of 16 hidden
// channels, the 16 gate rows followed by the 16 up rows (a last, shorter run is padded with zero rows), so that a tile
// of 64 output columns holds gate and up products of the same 32 channels:  g = min(gate, limit),
// u = clamp(up, -limit, limit);  hidden = g * sigmoid(alpha * g) * (u + shift).
struct GluParams {
  float alpha, limit, shift;
};
__device__ __forceinline__ float clamped_glu(float gate, float up, const GluParams& p) {
  const float g = fminf(gate, p.limit), u = fminf(fmaxf(up, -p.limit), p.limit);
  return g * sigmoidf_(p.alpha * g) * (u + p.shift);
}

// -> expert and first sorted row of this workgroup's tile of `tm` rows, rows in it (0: nothing to do)
__device__ __forceinline__ int find_tile(const int32_t* __restrict__ expert_start, int num_experts, int tile,
                                         int* expert, int* row0, int tm = TM) {
  for (int e = 0; e < num_experts; ++e) {
    const int lo = expert_start[e], n = expert_start[e + 1] - lo;
    const int tiles = (n + tm - 1) / tm;
    if (tile < tiles) {
      *expert = e;
      *row0 = lo + tile * tm;
      return min(tm, n - tile * tm);
    }
    tile -= tiles;
  }
  return 0;
}

template <typename T>
__global__ __launch_bounds__(kFfnThreads) void expert_up_gelu_kernel(
    void* __restrict__ hidden, const void* __restrict__ x, const void* __restrict__ up,
    const int32_t* __restrict__ order, const int32_t* __restrict__ expert_start, int num_experts, int width, int ff,
    int top, int activation, int up_rows, GluParams glu, const float* __restrict__ pair_weight) {
  __shared__ float As[TM][TK + 1];
  __shared__ float Bs[TN][TK + 1];
  int e, row0;
  const int rows = find_tile(expert_start, num_experts, blockIdx.x, &e, &row0);
  if (rows == 0) return;
  const int n0 = blockIdx.y * TN;
  float acc[2][4];
  tile_gemm<T>(acc, x, [&](int r) { return (int64_t)(order[row0 + r] / top) * width; }, rows, up, (int64_t)e * up_rows * width, n0,
               up_rows, width, As, Bs);
  const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 2 * ty + i;
    if (r >= rows) continue;
    if (pair_weight != nullptr) {                            // the weight of the expert's INPUT, taken through the products
      const float wt = pair_weight[order[row0 + r]];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] *= wt;
    }
    if (activation == SWM_ACT_CLAMPED_GLU) {
      // columns tx + 16 j of the tile: j = 0, 2 are gate products, j = 1, 3 the up products of the same channels
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const int ch = (n0 / 32 + j / 2) * 16 + tx;
        if (ch < ff) st<T>(hidden, (int64_t)(row0 + r) * ff + ch, clamped_glu(acc[i][j], acc[i][j + 1], glu));
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx + 16 * j;
      if (n < ff) st<T>(hidden, (int64_t)(row0 + r) * ff + n, expert_act(acc[i][j], activation));
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kFfnThreads) void expert_down_kernel(
    float* __restrict__ out, const void* __restrict__ hidden, const void* __restrict__ down,
    const int32_t* __restrict__ order, const int32_t* __restrict__ expert_start, int num_experts, int width, int ff,
    int top, float weight, const float* __restrict__ pair_weight) {
  __shared__ float As[TM][TK + 1];
  __shared__ float Bs[TN][TK + 1];
  int e, row0;
  const int rows = find_tile(expert_start, num_experts, blockIdx.x, &e, &row0);
  if (rows == 0) return;
  const int n0 = blockIdx.y * TN;
  float acc[2][4];
  tile_gemm<T>(acc, hidden, [&](int r) { return (int64_t)(row0 + r) * ff; }, rows, down, (int64_t)e * width * ff, n0, width,
               ff, As, Bs);
  const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 2 * ty + i;
    if (r >= rows) continue;
    const int pair = order[row0 + r];
    const int64_t dst = pair / top;
    const float wt = pair_weight != nullptr ? weight * pair_weight[pair] : weight;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx + 16 * j;
      if (n >= width) continue;
      float* p = out + dst * width + n;
      if (top == 1) *p += wt * acc[i][j];               // a row has one expert: nobody else writes it
      else atomicAdd(p, wt * acc[i][j]);
    }
  }
}


// ------------------------------------------------------------------------------- bf16 on the matrix cores
// Both kernels compute  up: hidden[pair] = act(up[e] x[row])  and  down: out[row] += weight * down[e] hidden[pair]  for the
// pairs of one expert; DOWN picks the operands and the epilogue.
struct ExpertArgs {
  void* out;                            // up: bf16 hidden [pairs, ff]; down: fp32 [rows, width]
  const uint16_t *x, *w;                // up: x [rows, K], up [E, N, K]; down: hidden [pairs, K], down [E, N, K]
  const int32_t *order, *expert_start;
  const float* pair_weight;
  int num_experts, K, N, ff, top, activation;
  float weight;
  GluParams glu;
};
using f32x4 = __attribute__((ext_vector_type(4))) float;
using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;

// four neighbouring channels of one pair's hidden layer
__device__ __forceinline__ void store_hidden(const ExpertArgs& a, int64_t sorted_row, int ch, const float (&v)[4]) {
  const int64_t at = sorted_row * a.ff + ch;
  if (a.ff % 4 == 0) {
    if (ch < a.ff) st_vec<sw::bf16_t, 4>(a.out, at, v);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (ch + j < a.ff) st<sw::bf16_t>(a.out, at + j, v[j]);
  }
}

// Steps of few rows per expert (decode steps): what bounds them is the experts' weights, which must stream at memory speed.
// A workgroup owns 32 weight rows of one expert; its 4 waves share the reduction out among them and every wave reads its part
// of the rows straight into the A operand of v_mfma_f32_16x16x32_bf16 (16 rows, 8 neighbouring k per lane), 16 loads in
// flight per lane before the first product, no barrier before the waves' sums meet in LDS.  The pairs are the B operand, up
// to 32 at a time (PT tiles of 16), so weights are read once per 32 pairs.
// C element r of lane l: weight row 4 (l / 16) + r, pair l % 16.
// Measured, 61 rows of width 2048, 32 gated experts of 1024, two per row (396 MB of weights), sort and clearing included:
// 120 us in tiles of 64 x 64 with a load, a barrier and a product in turn, 81 us here (4.9 TB/s; 5.8 without the sort).
constexpr int kFewRows = 32, kFewWaves = 4;

template <bool DOWN, int PT>
__device__ __forceinline__ void few_rows_pass(const ExpertArgs& a, int e, int64_t lo, int p0, int n, int n0, float* red) {
  constexpr int U = PT == 1 ? 8 : 4;                         // k steps whose operands are asked for together
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, kq = (lane >> 4) * 8;
  const uint16_t* wp[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    wp[i] = a.w + ((int64_t)e * a.N + min(n0 + 16 * i + li, a.N - 1)) * a.K + kq;
  const uint16_t* xp[PT];
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    const int64_t row = lo + min(p0 + 16 * j + li, n - 1);
    xp[j] = a.x + (DOWN ? row : (int64_t)(a.order[row] / a.top)) * a.K + kq;
  }
  f32x4 acc[PT][2];
#pragma unroll
  for (int j = 0; j < PT; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) acc[j][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int steps = (a.K + 31) / 32, share = (steps + kFewWaves - 1) / kFewWaves;
  int s = wave * share;
  const int s_end = min(steps, s + share), s_full = min(s_end, a.K / 32);
  for (; s + U <= s_full; s += U) {
    bf16x8 wf[U][2], xf[U][PT];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) wf[u][i] = *reinterpret_cast<const bf16x8*>(wp[i] + (s + u) * 32);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < PT; ++j) xf[u][j] = *reinterpret_cast<const bf16x8*>(xp[j] + (s + u) * 32);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < PT; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][i], xf[u][j], acc[j][i], 0, 0, 0);
  }
  for (; s < s_end; ++s) {                                   // the rest, the last step perhaps of less than 32
    const bool in = s * 32 + kq < a.K;
    union { u32x4 w; bf16x8 v; } wf[2], xf;
#pragma unroll
    for (int i = 0; i < 2; ++i) wf[i].w = in ? *reinterpret_cast<const u32x4*>(wp[i] + s * 32) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      xf.w = in ? *reinterpret_cast<const u32x4*>(xp[j] + s * 32) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i].v, xf.v, acc[j][i], 0, 0, 0);
    }
  }
  // ---- the waves' sums, in a fixed order; wave j % 4 finishes tile j
  f32x4* mine = reinterpret_cast<f32x4*>(red);
#pragma unroll
  for (int j = 0; j < PT; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) mine[((wave * PT + j) * 2 + i) * 64 + lane] = acc[j][i];
  __syncthreads();
  if (wave < PT) {
    const int j = wave, p = p0 + 16 * j + li;
    f32x4 sum[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      sum[i] = mine[(j * 2 + i) * 64 + lane];
#pragma unroll
      for (int w = 1; w < kFewWaves; ++w) sum[i] += mine[((w * PT + j) * 2 + i) * 64 + lane];
    }
    if (p < n) {
      const int c4 = 4 * (lane >> 4);
      const int pair = a.order[lo + p];
      if constexpr (!DOWN) {
        const float wt = a.pair_weight != nullptr ? a.pair_weight[pair] : 1.0f;
        if (a.activation == SWM_ACT_CLAMPED_GLU) {           // rows 0..15 of the 32 are gates, 16..31 the same channels' ups
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = clamped_glu(sum[0][r] * wt, sum[1][r] * wt, a.glu);
          store_hidden(a, lo + p, n0 / 2 + c4, v);
        } else {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = expert_act(sum[i][r] * wt, a.activation);
            store_hidden(a, lo + p, n0 + 16 * i + c4, v);
          }
        }
      } else {
        const float wt = a.pair_weight != nullptr ? a.weight * a.pair_weight[pair] : a.weight;
        float* dst = static_cast<float*>(a.out) + (int64_t)(pair / a.top) * a.N;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int c = n0 + 16 * i + c4 + r;
            if (c < a.N) atomicAdd(dst + c, wt * sum[i][r]);
          }
      }
    }
  }
  __syncthreads();
}

template <bool DOWN>
__global__ __launch_bounds__(64 * kFewWaves) void expert_few_rows_kernel(const ExpertArgs a) {
  __shared__ __attribute__((aligned(16))) float red[kFewWaves * 2 * 2 * 64 * 4];
  const int e = blockIdx.y, lo = a.expert_start[e], n = a.expert_start[e + 1] - lo, n0 = blockIdx.x * kFewRows;
  for (int p0 = blockIdx.z * 32; p0 < n; p0 += gridDim.z * 32) {         // uniform over the workgroup
    if (n - p0 <= 16) few_rows_pass<DOWN, 1>(a, e, lo, p0, n, n0, red);
    else few_rows_pass<DOWN, 2>(a, e, lo, p0, n, n0, red);
  }
}

// Steps of more rows per expert (prompt steps): matrix work.  A workgroup of 4 waves computes BM pairs x BN weight rows of one
// expert, (BM / 2) x (BN / 2) per wave (v_mfma_f32_32x32x16_bf16); stages of 64 k go global -> registers three stages ahead
// (two register sets in turn) and registers -> LDS one stage ahead, one barrier a stage; the order of LDS reads and products
// inside a stage is pinned, half of the reads before the first product.
// Workgroup numbers go round-robin over the 8 XCDs, each with an L2 of its own: an XCD takes a contiguous part of the tiles in
// the order (expert, weight rows, pairs), so an expert's pairs stay in one L2 and a block of weights is read by workgroups
// that follow one another there.
// Measured, 3989 rows of width 2048, 32 gated experts of 1024, two per row (7978 pairs), up / down: 287 / 188 us in the 64 x 64
// tiles with a load, a barrier and a product in turn that these replace; 168 / 119 us with 128 x 128 tiles whose loads were
// one stage ahead; 134 / 109 us as it is (498 / 308 TFLOP/s; one by one under a profiler, 5 % less in a stream of calls).  Of the
// down-projection 26 us are its additions into the fp32 output (plain stores instead: 82 us).
constexpr int kTileK = 64, kTilePad = 8;
__host__ __device__ constexpr int expert_tile_lds(int tm, int tn) { return 2 * (tm + tn) * (kTileK + kTilePad) * 2 + 2 * tm * 4; }

// WHOLE: K is a multiple of 64.
template <bool DOWN, int BM, int BN, bool WHOLE>
__global__ __launch_bounds__(256, 2) void expert_tile_kernel(const ExpertArgs a) {
  extern __shared__ __attribute__((aligned(16))) char big_lds[];
  constexpr int STRIDE = kTileK + kTilePad;
  uint16_t* Xs = reinterpret_cast<uint16_t*>(big_lds);                   // [2][BM][STRIDE]
  uint16_t* Ws = Xs + 2 * BM * STRIDE;                                   // [2][BN][STRIDE]
  int* pair_of = reinterpret_cast<int*>(Ws + 2 * BN * STRIDE);           // [BM]
  float* weight_of = reinterpret_cast<float*>(pair_of + BM);             // [BM]
  constexpr int XL = BM / 32, WL = BN / 32;                              // pieces that a thread stages
  constexpr int MI = BM / 64, NI = BN / 64;                              // accumulators of a wave
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // ---- which tile: lane l of a wave looks at expert l of every 64
  const int cols = (a.N + BN - 1) / BN;
  int row_tiles = 0;
  for (int e0 = 0; e0 < a.num_experts; e0 += 64) {
    const int ex = e0 + lane;
    int tiles = ex < a.num_experts ? (a.expert_start[ex + 1] - a.expert_start[ex] + BM - 1) / BM : 0;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) tiles += __shfl_xor(tiles, m, 64);
    row_tiles += tiles;
  }
  const int64_t total = (int64_t)row_tiles * cols, per = (total + 7) / 8;
  const int64_t local = blockIdx.x >> 3;
  int64_t t = (blockIdx.x & 7) * per + local;
  if (local >= per || t >= total) return;                    // the whole workgroup
  int e = -1, lo = 0, n = 0, rt = 0, ct = 0;
  for (int e0 = 0; e0 < a.num_experts; e0 += 64) {
    const int ex = e0 + lane;
    const int first = ex < a.num_experts ? a.expert_start[ex] : 0;
    const int count = ex < a.num_experts ? a.expert_start[ex + 1] - first : 0;
    const int tiles = (count + BM - 1) / BM;
    int upto = tiles;                                        // tiles of the experts up to this lane's
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const int o = __shfl_up(upto, m, 64);
      if (lane >= m) upto += o;
    }
    const uint64_t past = __builtin_amdgcn_ballot_w64((int64_t)upto * cols > t);
    if (past != 0) {
      const int l = __builtin_ctzll(past);
      const int mine = __shfl(tiles, l, 64);
      const int rem = (int)(t - (int64_t)(__shfl(upto, l, 64) - mine) * cols);
      e = e0 + l;
      lo = __shfl(first, l, 64);
      n = __shfl(count, l, 64);
      ct = rem / mine;
      rt = rem - ct * mine;
      break;
    }
    t -= (int64_t)__shfl(upto, 63, 64) * cols;
  }
  e = __builtin_amdgcn_readfirstlane(e);
  lo = __builtin_amdgcn_readfirstlane(lo);
  n = __builtin_amdgcn_readfirstlane(n);
  rt = __builtin_amdgcn_readfirstlane(rt);
  ct = __builtin_amdgcn_readfirstlane(ct);
  const int64_t row0 = lo + (int64_t)rt * BM;          // first sorted pair
  const int rows = min(BM, n - rt * BM), n0 = ct * BN;
  if (tid < BM) {
    const int pair = a.order[row0 + min(tid, rows - 1)];
    pair_of[tid] = pair;
    weight_of[tid] = a.pair_weight != nullptr ? a.pair_weight[pair] : 1.0f;
  }

  // ---- staging: rows tid / 8 + 32 i, piece tid % 8 of 16 bytes (rows beyond the tile repeat its last one)
  const int ch = (tid & 7) * 8;
  const uint16_t *xp[XL], *wp[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int64_t row = row0 + min((tid >> 3) + 32 * i, rows - 1);
    xp[i] = a.x + (DOWN ? row : (int64_t)(a.order[row] / a.top)) * a.K;
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) wp[i] = a.w + ((int64_t)e * a.N + min(n0 + (tid >> 3) + 32 * i, a.N - 1)) * a.K;
  // Two register sets take turns, so a stage's loads have two stages of matrix work to land.  Every stage issues the same
  // loads (past the end: the last stage's again), or the compiler could not count what is in flight and would wait for all.
  u32x4 xr[2][XL], wr[2][WL];
  const int stages = (a.K + kTileK - 1) / kTileK;
  auto fetch = [&](auto SET, int s) {
    constexpr int set = decltype(SET)::value;
    const int k = min(min(s, stages - 1) * kTileK + ch, a.K - 8);        // K is a multiple of 8
    sw::static_for<XL>([&](auto I) { xr[set][decltype(I)::value] = *reinterpret_cast<const u32x4*>(xp[decltype(I)::value] + k); });
    sw::static_for<WL>([&](auto I) { wr[set][decltype(I)::value] = *reinterpret_cast<const u32x4*>(wp[decltype(I)::value] + k); });
  };
  auto commit = [&](auto SET, int s, int buf) {
    constexpr int set = decltype(SET)::value;
    if (!WHOLE && s == stages - 1 && s * kTileK + ch >= a.K) {           // a last stage of less than 64
      sw::static_for<XL>([&](auto I) { xr[set][decltype(I)::value] = u32x4{0u, 0u, 0u, 0u}; });
      sw::static_for<WL>([&](auto I) { wr[set][decltype(I)::value] = u32x4{0u, 0u, 0u, 0u}; });
    }
    sw::static_for<XL>([&](auto I) {
      constexpr int i = decltype(I)::value;
      *reinterpret_cast<u32x4*>(Xs + (buf * BM + (tid >> 3) + 32 * i) * STRIDE + ch) = xr[set][i];
    });
    sw::static_for<WL>([&](auto I) {
      constexpr int i = decltype(I)::value;
      *reinterpret_cast<u32x4*>(Ws + (buf * BN + (tid >> 3) + 32 * i) * STRIDE + ch) = wr[set][i];
    });
  };
  const int wm = wave >> 1, wn = wave & 1, li = lane & 31, hl = lane >> 5;
  f32x16 acc[MI][NI];                                        // [32 pairs][32 weight rows]
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  fetch(Even{}, 0);
  __builtin_amdgcn_sched_barrier(0);
  fetch(Odd{}, 1);
  __builtin_amdgcn_sched_barrier(0);
  commit(Even{}, 0, 0);
  fetch(Even{}, 2);
  __syncthreads();
  // stage s: stage s + 1 registers -> LDS (the set that stage s + 3 is then asked into) | products of stage s | barrier
  auto stage = [&](auto NEXT, int s, int buf) {
    commit(NEXT, s + 1, buf ^ 1);
    fetch(NEXT, s + 3);
    __builtin_amdgcn_sched_barrier(0);                       // or the loads are moved behind the products
    const uint16_t* xb = Xs + (buf * BM + wm * (BM / 2) + li) * STRIDE + 8 * hl;
    const uint16_t* wb = Ws + (buf * BN + wn * (BN / 2) + li) * STRIDE + 8 * hl;
    constexpr int KS = kTileK / 16, READS = KS * (MI + NI), PRODUCTS = KS * MI * NI;
    bf16x8 xf[KS][MI], wf[KS][NI];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int i = 0; i < MI; ++i) xf[ks][i] = *reinterpret_cast<const bf16x8*>(xb + 32 * i * STRIDE + 16 * ks);
#pragma unroll
      for (int j = 0; j < NI; ++j) wf[ks][j] = *reinterpret_cast<const bf16x8*>(wb + 32 * j * STRIDE + 16 * ks);
    }
    // up: C rows are weight rows (a lane ends up with neighbouring channels of one pair, gates beside their ups);
    // down: C columns are (a wave's lanes add to neighbouring channels of one row)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[i][j] = DOWN ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[ks][i], wf[ks][j], acc[i][j], 0, 0, 0)
                           : __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[ks][j], xf[ks][i], acc[i][j], 0, 0, 0);
    // half of the LDS reads before the first product, the others spread among the products
    __builtin_amdgcn_sched_group_barrier(0x100, READS / 2, 0);
#pragma unroll
    for (int u = 0; u < PRODUCTS / 2; ++u) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, READS / PRODUCTS, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, PRODUCTS / 2, 0);
    __syncthreads();
  };
  // (no condition inside the loop: what is in flight has to be the same on every way to a wait)
  int s = 0;
#pragma unroll 1
  for (; s + 1 < stages; s += 2) {
    stage(Odd{}, s, 0);
    stage(Even{}, s + 1, 1);
  }
  if (s < stages) stage(Odd{}, s, 0);
  // C element r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32
  if constexpr (!DOWN) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int p = wm * (BM / 2) + 32 * i + li;
      if (p >= rows) continue;
      const float wt = weight_of[p];
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int c0 = n0 + wn * (BN / 2) + 32 * j;
        if (a.activation == SWM_ACT_CLAMPED_GLU) {           // rows 0..15 of every 32 are gates, 16..31 the channels' ups
#pragma unroll
          for (int r4 = 0; r4 < 2; ++r4) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
              v[r] = clamped_glu(acc[i][j][4 * r4 + r] * wt, acc[i][j][8 + 4 * r4 + r] * wt, a.glu);
            store_hidden(a, row0 + p, c0 / 2 + 8 * r4 + 4 * hl, v);
          }
        } else {
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = expert_act(acc[i][j][4 * r4 + r] * wt, a.activation);
            store_hidden(a, row0 + p, c0 + 8 * r4 + 4 * hl, v);
          }
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int p = wm * (BM / 2) + 32 * i + 8 * (r / 4) + 4 * hl + r % 4;
        if (p >= rows) continue;
        const float wt = a.weight * weight_of[p];
        float* dst = static_cast<float*>(a.out) + (int64_t)(pair_of[p] / a.top) * a.N;
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const int c = n0 + wn * (BN / 2) + 32 * j + li;
          if (c < a.N) atomicAdd(dst + c, wt * acc[i][j][r]);
        }
      }
  }
}

template <bool DOWN, int BM, int BN, bool WHOLE>
int launch_expert_tiles_as(const ExpertArgs& a, int64_t pairs, hipStream_t stream) {
  const int64_t tiles = ((pairs + BM - 1) / BM + a.num_experts) * ((a.N + BN - 1) / BN);           // an upper bound
  SW_CHECK_ARG(tiles < (1ll << 31) - 8, "expert_ffn: too many tiles");
  constexpr int lds = expert_tile_lds(BM, BN);
  if (lds > 64 * 1024)
    SW_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(expert_tile_kernel<DOWN, BM, BN, WHOLE>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  hipLaunchKernelGGL((expert_tile_kernel<DOWN, BM, BN, WHOLE>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), lds, stream, a);
  SW_CHECK_LAUNCH();
  return SW_OK;
}

template <bool DOWN, int BM, int BN>
int launch_expert_tiles(const ExpertArgs& a, int64_t pairs, hipStream_t stream) {
  return a.K % kTileK == 0 ? launch_expert_tiles_as<DOWN, BM, BN, true>(a, pairs, stream)
                           : launch_expert_tiles_as<DOWN, BM, BN, false>(a, pairs, stream);
}

// Which kernel: by the average number of pairs per expert (the host does not know the real one) and by the tiles that a
// launch has.  Measured (whole feed-forward with its sort and clearing, us; weights streamed / 64 x 64 tiles / 128 x 128 tiles /
// the 64 x 64 tiles of before):
//   32 gated experts 2048 -> 1024:   2 pairs each 78 / 87 / 87 / 114;   6: 89 / 90 / 94 / 125;   8: 95 / 93 / 98 / 133;
//                                    64: 231 / 130 / 146 / 187;   128: 386 / 174 / 168 / 281;   250: 711 / 272 / 226 / 473
//   64 experts 2048 -> 1024, four per row:  6: 114 / 115 / 120 / 149;   96: 432 / 200 / 197 / 311;   250: 994 / 365 / 308 / 640
//   8 experts 2048 -> 1024, 250 pairs each: 148 / 64 / 70 / 108: too few tiles of 128 x 128 for 256 compute units
constexpr int kFewPairs = 6;            // pairs per expert up to which a step's weights are streamed
constexpr int kFewGroups = 16384;      // workgroups of such a launch, of which most may find nothing to do
constexpr int kManyPairs = 96;          // pairs per expert from which tiles of 128 pairs are mostly full ...
constexpr int kManyTiles = 384;         // ... if there are this many of them
template <bool DOWN>
int launch_experts(const ExpertArgs& a, int64_t pairs, hipStream_t stream) {
  if (pairs <= (int64_t)kFewPairs * a.num_experts && a.num_experts < 65536) {
    // an expert that many more rows ask for than the average has its rows shared out among several workgroups: one for every 64
    // pairs where the launch stays within kFewGroups workgroups, or else for every 256 (most of them find nothing to do).  64 experts
    // 2048 -> 1024, all of 200 rows on one: 91 us in 64 x 64 tiles, 111 with a workgroup for all, 77 with 4
    const int64_t cols = (a.N + kFewRows - 1) / kFewRows;
    const int64_t room = std::max<int64_t>(std::min<int64_t>(8, (pairs + 255) / 256), kFewGroups / (cols * a.num_experts));
    const unsigned shares = (unsigned)std::min<int64_t>(room, (pairs + 63) / 64);
    const dim3 grid((unsigned)cols, (unsigned)a.num_experts, shares);
    hipLaunchKernelGGL(expert_few_rows_kernel<DOWN>, grid, dim3(64 * kFewWaves), 0, stream, a);
    SW_CHECK_LAUNCH();
    return SW_OK;
  }
  const int64_t big_tiles = pairs / 128 * ((a.N + 127) / 128);
  if (pairs >= (int64_t)kManyPairs * a.num_experts && big_tiles >= kManyTiles)
    return launch_expert_tiles<DOWN, 128, 128>(a, pairs, stream);
  return launch_expert_tiles<DOWN, 64, 64>(a, pairs, stream);
}

}  // namespace swm

extern "C" {

int swm_expert_up_gelu(void* hidden, const void* x, const void* up, const int32_t* order,
                       const int32_t* expert_start, int num_experts, int64_t sorted_rows, int width, int ff,
                       int top, int act_dtype, void* stream) {
  return swm_expert_up(hidden, x, up, order, expert_start, num_experts, sorted_rows, width, ff, top, SWM_ACT_GELU,
                       act_dtype, stream);
}

int swm_expert_up(void* hidden, const void* x, const void* up, const int32_t* order, const int32_t* expert_start,
                  int num_experts, int64_t sorted_rows, int width, int ff, int top, int activation, int act_dtype,
                  void* stream) {
  return swm_expert_up_as(hidden, x, up, order, expert_start, num_experts, sorted_rows, width, ff, top, activation, 1.0f,
                          INFINITY, 0.0f, act_dtype, stream);
}

int swm_expert_up_as(void* hidden, const void* x, const void* up, const int32_t* order, const int32_t* expert_start,
                     int num_experts, int64_t sorted_rows, int width, int ff, int top, int activation, float glu_alpha,
                     float glu_limit, float glu_shift, int act_dtype, void* stream) {
  return swm_expert_up_weighted(hidden, x, up, order, expert_start, num_experts, sorted_rows, width, ff, top, activation,
                                glu_alpha, glu_limit, glu_shift, nullptr, act_dtype, stream);
}

int swm_expert_up_weighted(void* hidden, const void* x, const void* up, const int32_t* order,
                           const int32_t* expert_start, int num_experts, int64_t sorted_rows, int width, int ff, int top,
                           int activation, float glu_alpha, float glu_limit, float glu_shift, const float* pair_weight,
                           int act_dtype, void* stream) {
  using namespace swm;
  if (sorted_rows == 0) return SW_OK;
  const bool gated = activation == SWM_ACT_CLAMPED_GLU;
  const int up_rows = gated ? 32 * ((ff + 15) / 16) : ff;     // runs of 16 gate rows + 16 up rows
  const GluParams glu{glu_alpha, glu_limit, glu_shift};
  SW_CHECK_ARG(activation == SWM_ACT_GELU || activation == SWM_ACT_RELU2 || activation == SWM_ACT_NONE || gated,
               "expert_up: unknown activation %d", activation);
  SW_CHECK_ARG(act_ok(act_dtype), "expert_up_gelu: unsupported dtype %d", act_dtype);
  SW_CHECK_ARG(num_experts > 0 && width > 0 && ff > 0 && top > 0 && sorted_rows < (1ll << 30), "expert_up_gelu: bad shape");
  if (act_dtype == SW_BF16 && width % 8 == 0) {
    ExpertArgs a{hidden, static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(up), order, expert_start, pair_weight,
                 num_experts, width, up_rows, ff, top, activation, 1.0f, glu};
    return launch_experts<false>(a, sorted_rows, static_cast<hipStream_t>(stream));
  }
  const dim3 grid((unsigned)((sorted_rows + TM - 1) / TM + num_experts), (unsigned)((up_rows + TN - 1) / TN));
  SWM_DISPATCH_ACT(act_dtype, hipLaunchKernelGGL(expert_up_gelu_kernel<T>, grid, dim3(kFfnThreads), 0,
                                                 static_cast<hipStream_t>(stream), hidden, x, up, order, expert_start,
                                                 num_experts, width, ff, top, activation, up_rows, glu, pair_weight););
  SW_CHECK_LAUNCH();
  return SW_OK;
}

int swm_expert_down(float* out, const void* hidden, const void* down, const int32_t* order,
                    const int32_t* expert_start, int num_experts, int64_t sorted_rows, int width, int ff,
                    int top, float weight, int act_dtype, void* stream) {
  return swm_expert_down_weighted(out, hidden, down, order, expert_start, num_experts, sorted_rows, width, ff, top,
                                  weight, nullptr, act_dtype, stream);
}

int swm_expert_down_weighted(float* out, const void* hidden, const void* down, const int32_t* order,
                             const int32_t* expert_start, int num_experts, int64_t sorted_rows, int width, int ff,
                             int top, float weight, const float* pair_weight, int act_dtype, void* stream) {
  using namespace swm;
  if (sorted_rows == 0) return SW_OK;
  SW_CHECK_ARG(act_ok(act_dtype), "expert_down: unsupported dtype %d", act_dtype);
  SW_CHECK_ARG(num_experts > 0 && width > 0 && ff > 0 && top > 0 && sorted_rows < (1ll << 30), "expert_down: bad shape");
  if (act_dtype == SW_BF16 && ff % 8 == 0) {
    ExpertArgs a{out, static_cast<const uint16_t*>(hidden), static_cast<const uint16_t*>(down), order, expert_start, pair_weight,
                 num_experts, ff, width, ff, top, SWM_ACT_NONE, weight, GluParams{1.0f, INFINITY, 0.0f}};
    return launch_experts<true>(a, sorted_rows, static_cast<hipStream_t>(stream));
  }
  const dim3 grid((unsigned)((sorted_rows + TM - 1) / TM + num_experts), (unsigned)((width + TN - 1) / TN));
  SWM_DISPATCH_ACT(act_dtype, hipLaunchKernelGGL(expert_down_kernel<T>, grid, dim3(kFfnThreads), 0,
                                                 static_cast<hipStream_t>(stream), out, hidden, down, order,
                                                 expert_start, num_experts, width, ff, top, weight, pair_weight););
  SW_CHECK_LAUNCH();
  return SW_OK;
}

}  // extern "C"
