// Decode steps of the paged attention in capped_attention.hip over a bf16 cache: at most 8 query rows (tokens x query heads of a
// group) per sequence and key/value head, on the bf16 matrix cores with fp32 scores and weights (prompt_attention.hip tells why
// three bf16 products of an operand's exact parts are the fp32 product).
//
// What bounds it: the cache's way from memory, so the work beside it has to be small and the loads have to stay in flight.
//   * The parts of FOUR query rows lie side by side in the 16 columns of one operand (column 4 part + row): one
//     v_mfma_f32_16x16x32_bf16 makes the products of all three parts with 16 keys x 32 coordinates, and two rotations within
//     the rows of 16 lanes add them up, in every lane.  Eight rows take two such sets.
//   * S^T = K Q^T: A = keys, straight from the cache into registers (lane l: key l % 16, 8 neighbouring coordinates).
//     C element r of lane l: key 4 (l / 16) + r, column l % 16.
//   * O^T = V^T P^T: two key tiles' C registers are the B operand's 8 keys per lane; each lane keeps of its weights the part that
//     its column stands for.  A comes from a row-major stage in LDS, the wave's own, by the transposing ds_read_b64_tr_b16.
//   * A wave walks tiles of 32 keys by itself: 16 KB of keys and values are on their way while it works on the tile before
//     (page numbers two tiles ahead); no barrier until the waves are joined, in a fixed order.
// The output is referred to a new running maximum only when some lane's has grown by more than e^5.5, so a weight is below 2^8.
// A row that comes out as NaN is worked out again in fp32 (plain_row): a part that is zero, as a fourth of the columns is, makes NaN of
// an infinity in the cache.
// Few sequences share each one's keys out among `parts` workgroups, joined by a second kernel.
//
// Measured, 61 sequences of about 2041 keys (257 MB), 16 query heads on 4 of size 128: 100 us on the vector units (8 lanes per
// key, loads and arithmetic in turn), 61 us here; 55 us with the loads alone, streaming hints change nothing.  At 514 MB 112 us
// (4.6 TB/s) and 104.  Two sequences of 3000 keys: 21 us together with the join, in 16 parts each.
#include "prompt_attention.cuh"

#include <algorithm>

namespace swm {

using da_bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using da_f32x4 = __attribute__((ext_vector_type(4))) float;
using da_u32x4 = __attribute__((ext_vector_type(4))) uint32_t;
using da_i16x4 = __attribute__((ext_vector_type(4))) short;
using da_lds_i16x4 = __attribute__((address_space(3))) da_i16x4*;

constexpr int kDaKeys = 32, kDaWaves = 8;
constexpr float kDaLog2e = 1.4426950408889634f, kDaGrowth = 5.5f;                    // e^5.5 < 2^8
__device__ __forceinline__ float da_exp(float x) { return __builtin_amdgcn_exp2f(x * kDaLog2e); }

union DaFrag {
  uint32_t w[4];
  da_bf16x8 v;
};

__host__ __device__ constexpr int da_vstride(int nb) { return nb * 64 + 32; }        // bytes of a staged value row
__host__ __device__ constexpr int da_lds_bytes(int nb) { return kDaWaves * (kDaKeys * da_vstride(nb) + 8 * 2 * 4 + kPlainRowLds * 4); }

// part `part` of x = h + m + l (truncated to bf16 one after the other: exact), in the upper half; 0: h, 1: m, 3: l, 2: nothing.  An infinity or NaN
// stays whole in h.  (A weight is at most 2^8: no infinity, and a NaN may spread.)
template <bool WEIGHT>
__device__ __forceinline__ uint32_t da_part(float x, int part) {
  const uint32_t h = __float_as_uint(x) & 0xffff0000u;
  const float r1 = !WEIGHT && (h & 0x7f800000u) == 0x7f800000u ? 0.0f : x - __uint_as_float(h);
  const uint32_t m = __float_as_uint(r1) & 0xffff0000u;
  const uint32_t l = __float_as_uint(r1 - __uint_as_float(m));
  return part == 0 ? h : part == 1 ? m : part == 3 ? l : 0u;
}
__device__ __forceinline__ uint32_t da_upper_halves(uint32_t hi, uint32_t lo) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); }
// x rotated by N lanes within the rows of 16 lanes
template <int N>
__device__ __forceinline__ float da_rotated(float x) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x120 + N, 0xf, 0xf, false));
}
// the sum over the columns of a query row, in all of them: h + (m + l), one rounding that counts
__device__ __forceinline__ float da_parts_sum(float x) {
  x += da_rotated<8>(x);
  return x + da_rotated<4>(x);
}
// over the four rows of 16 lanes
__device__ __forceinline__ float da_rows_max(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float da_rows_sum(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// NB: blocks of 32 coordinates of the larger of key and value size.  NS: sets of four query rows.
template <int NB, int NS>
__global__ __launch_bounds__(64 * kDaWaves, 2) void decode_attention_kernel(const PromptAttention a, float* __restrict__ partial,
                                                                            int64_t total_rows) {
  constexpr int VSTRIDE = da_vstride(NB), CPR = 4 * NB, VL = 2 * NB;
  extern __shared__ __attribute__((aligned(16))) char da_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, g16 = lane >> 4, part = c16 >> 2, qr = c16 & 3;
  char* stage = da_lds + wave * kDaKeys * VSTRIDE;                                   // [32][VSTRIDE]; later [rows][32 NB] floats
  float* Ml = reinterpret_cast<float*>(da_lds + kDaWaves * kDaKeys * VSTRIDE);       // [waves][8][2]; then the plain rows' floats
  const int seq = blockIdx.x, g = blockIdx.y, R = a.heads / a.kv_heads;
  const int row0 = a.q_start[seq], n = a.q_start[seq + 1] - row0;
  if (n <= 0) return;                                        // the whole workgroup
  const int ctx = a.ctx_len[seq], rows = n * R, last_pos = ctx + n - 1;
  const int32_t* table = a.block_tables + (int64_t)seq * a.table_width;
  auto low_of = [&](int pos) { return a.chunk > 0 ? pos / a.chunk * a.chunk : a.window > 0 ? pos - a.window + 1 : 0; };
  const int lowest = max(low_of(ctx), 0), first_tile = lowest / kDaKeys, last_tile = last_pos / kDaKeys;
  const int low_last = low_of(last_pos);

  // ---- queries, scaled, this column's part of them.  (Scores stay as they are, their differences go to the log2 domain: large
  // scores scaled by log2 e through the queries cost 1.1 - 1.3 times the error of the results.)
  const bool sig = a.score_bias != nullptr, capped = a.softcap > 0.0f;
  const float cap_in = capped ? 2.0f * kDaLog2e / a.softcap : 0.0f;
  DaFrag q[NS][NB];
  float bias[NS];
  int pos[NS], low[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const int r = 4 * i + qr, tt = r / R, hh = r - tt * R;
    pos[i] = ctx + min(tt, n - 1);                           // padding rows behave like the last token's
    low[i] = low_of(pos[i]);
    bias[i] = sig ? a.score_bias[g * R + hh] : 0.0f;
#pragma unroll
    for (int ks = 0; ks < NB; ++ks) {
      const int c = 32 * ks + 8 * g16;
      const bool ok = r < rows && c < a.dim;
      const float* p = a.q + (int64_t)(row0 + tt) * a.heads * a.dim + (int64_t)(g * R + hh) * a.dim + c;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float4 x = ok ? *reinterpret_cast<const float4*>(p + 4 * j) : make_float4(0.f, 0.f, 0.f, 0.f);
        q[i][ks].w[2 * j] = da_upper_halves(da_part<false>(x.y * a.scale, part), da_part<false>(x.x * a.scale, part));
        q[i][ks].w[2 * j + 1] = da_upper_halves(da_part<false>(x.w * a.scale, part), da_part<false>(x.z * a.scale, part));
      }
    }
  }

  // ---- loads: keys beyond the last one are the last one again (one row, and masked)
  auto key_of = [&](int tile) { return max(min(tile * kDaKeys + (lane & 31), last_pos), lowest); };
  auto page_of = [&](int tile) {
    const int key = key_of(tile);
    return table[a.page_shift >= 0 ? key >> a.page_shift : key / a.page_size];
  };
  auto slot_of = [&](int page, int tile) {
    const int key = key_of(tile);
    return page * a.page_size + (a.page_shift >= 0 ? key & (a.page_size - 1) : key % a.page_size);
  };
  const bool kfull = a.dim == 32 * NB;
  da_u32x4 kreg[2][NB], vreg[VL];
  auto fetch_keys = [&](int slot) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint32_t s = (uint32_t)__shfl(slot, 16 * t + c16, 64);
      const uint16_t* kp = a.key_cache + (int64_t)s * a.k_stride + (int64_t)g * a.dim;
#pragma unroll
      for (int ks = 0; ks < NB; ++ks)
        kreg[t][ks] = *reinterpret_cast<const da_u32x4*>(kp + min(32 * ks + 8 * g16, a.dim - 8));
    }
  };
  auto fetch_values = [&](int slot) {
#pragma unroll
    for (int it = 0; it < VL; ++it) {
      const int c = it * 64 + lane, key = c / CPR, ch = c % CPR;
      const uint32_t s = (uint32_t)__shfl(slot, key, 64);
      vreg[it] = *reinterpret_cast<const da_u32x4*>(a.value_cache + (int64_t)s * a.v_stride + (int64_t)g * a.vdim +
                                                    min(8 * ch, a.vdim - 8));
    }
  };

  da_f32x4 o[NS][2 * NB];
  float m_run[NS], l_part[NS];
  const da_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    m_run[i] = sig ? 0.0f : -INFINITY;
    l_part[i] = 0.0f;
#pragma unroll
    for (int b = 0; b < 2 * NB; ++b) o[i][b] = zero;
  }
  // transposing reads: lane 4 i + p of a row of 16 lanes names value row i, channels 4 p .. 4 p + 3 of a 4 x 16 block
  const char* tr = stage + (4 * g16 + (c16 >> 2)) * VSTRIDE + (c16 & 3) * 8;

  const int step = gridDim.z * kDaWaves;
  int tile = first_tile + blockIdx.z * kDaWaves + wave;
  if (tile <= last_tile) {                                   // wave-uniform
    int slot = slot_of(page_of(tile), tile);
    int page = page_of(tile + step);
    fetch_keys(slot);
    fetch_values(slot);
#pragma unroll 1
    for (; tile <= last_tile; tile += step) {
      const int k0 = tile * kDaKeys;
      // ---- S^T = K Q^T
      da_f32x4 s[NS][2];
#pragma unroll
      for (int i = 0; i < NS; ++i) s[i][0] = s[i][1] = zero;
#pragma unroll
      for (int ks = 0; ks < NB; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          DaFrag kf;
          *reinterpret_cast<da_u32x4*>(kf.w) = kreg[t][ks];
          if (!kfull && 32 * ks + 8 * g16 >= a.dim) kf.w[0] = kf.w[1] = kf.w[2] = kf.w[3] = 0u;
#pragma unroll
          for (int i = 0; i < NS; ++i) s[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf.v, q[i][ks].v, s[i][t], 0, 0, 0);
        }
      // ---- the next tile's keys, the page numbers of the one after it before them
      slot = slot_of(page, tile + step);
      page = page_of(tile + 2 * step);
      fetch_keys(slot);
      __builtin_amdgcn_sched_barrier(0);
      // ---- cap, mask, running softmax (this lane: row qr of each set, keys 16 t + 4 g16 + r)
      DaFrag p[NS];
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        float x[8];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) x[4 * t + r] = da_parts_sum(s[i][t][r]);
        if (capped) {
#pragma unroll
          for (int j = 0; j < 8; ++j)                        // cap * tanh(s / cap) = cap (1 - 2 / (1 + e^(2 s / cap)))
            x[j] = a.softcap - 2.0f * a.softcap * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x[j] * cap_in));
        }
        if (k0 + kDaKeys - 1 > ctx || k0 < low_last) {       // wave-uniform: something to mask
          const int hi = pos[i] - k0 - 4 * g16, lo = low[i] - k0 - 4 * g16;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int at = 16 * (j / 4) + j % 4;
            x[j] = at <= hi && at >= lo ? x[j] : -INFINITY;
          }
        }
        if (sig) {
#pragma unroll
          for (int j = 0; j < 8; ++j)                        // a hidden key: 1 / (1 + e^inf) = 0
            x[j] = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-(x[j] + bias[i]) * kDaLog2e));
        } else {
          float tmax = x[0];
#pragma unroll
          for (int j = 1; j < 8; ++j) tmax = fmaxf(tmax, x[j]);
          const float m_new = fmaxf(m_run[i], da_rows_max(tmax));
          if (__builtin_amdgcn_ballot_w64(m_new > m_run[i] + kDaGrowth) != 0) {
            const float alpha = da_exp(m_run[i] - (m_new == -INFINITY ? 0.0f : m_new));
            l_part[i] *= alpha;
#pragma unroll
            for (int b = 0; b < 2 * NB; ++b) o[i][b] *= alpha;
            m_run[i] = m_new;
          }
          const float m_use = m_run[i] == -INFINITY ? 0.0f : m_run[i];
          float sum = 0.0f;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            x[j] = da_exp(x[j] - m_use);
            sum += x[j];
          }
          l_part[i] += sum;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) p[i].w[j] = da_upper_halves(da_part<true>(x[2 * j + 1], part), da_part<true>(x[2 * j], part));
      }
      // ---- O^T += V^T P^T; the wave's LDS accesses are carried out in order
#pragma unroll
      for (int it = 0; it < VL; ++it) {
        const int c = it * 64 + lane, key = c / CPR, ch = c % CPR;
        *reinterpret_cast<da_u32x4*>(stage + key * VSTRIDE + ch * 16) = vreg[it];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      fetch_values(slot);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < 2 * NB; ++b) {
        union { da_i16x4 half[2]; da_bf16x8 f; } v;
        v.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((da_lds_i16x4)(tr + b * 32));
        v.half[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((da_lds_i16x4)(tr + 16 * VSTRIDE + b * 32));
#pragma unroll
        for (int i = 0; i < NS; ++i) o[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v.f, p[i].v, o[i][b], 0, 0, 0);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
  // ---- join the waves: the columns of a row hold the same sums, each stores a quarter of the channels
  float* Os = reinterpret_cast<float*>(stage);
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const float l = da_rows_sum(l_part[i]);
    if (g16 == 0 && part == 0) {
      Ml[(wave * 8 + 4 * i + qr) * 2] = m_run[i];
      Ml[(wave * 8 + 4 * i + qr) * 2 + 1] = l;
    }
#pragma unroll
    for (int b = 0; b < 2 * NB; ++b) {
      da_f32x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = da_parts_sum(o[i][b][r]);
      if (part == b % 4) *reinterpret_cast<da_f32x4*>(Os + (4 * i + qr) * 32 * NB + 16 * b + 4 * g16) = y;
    }
  }
  __syncthreads();
  for (int e0 = 64 * wave; e0 < rows * a.vdim; e0 += 64 * kDaWaves) {                // uniform over the wave
    const int e = min(e0 + lane, rows * a.vdim - 1), r = e / a.vdim, c = e - r * a.vdim, tt = r / R, hh = r - tt * R;
    float m_all = -INFINITY;
#pragma unroll
    for (int w = 0; w < kDaWaves; ++w) m_all = fmaxf(m_all, Ml[(w * 8 + r) * 2]);
    const float sk = a.sink_logit != nullptr ? a.sink_logit[g * R + hh] : 0.0f;
    const bool sink = partial == nullptr && a.sink;
    float m_use = sink ? fmaxf(m_all, sk) : m_all;
    m_use = m_use == -INFINITY ? 0.0f : m_use;               // (a part that saw no key)
    float num = 0.0f, den = 0.0f;
#pragma unroll
    for (int w = 0; w < kDaWaves; ++w) {
      const float f = da_exp(Ml[(w * 8 + r) * 2] - m_use);
      den += f * Ml[(w * 8 + r) * 2 + 1];
      num += f * reinterpret_cast<const float*>(da_lds + w * kDaKeys * VSTRIDE)[r * 32 * NB + c];
    }
    for (uint64_t left = __builtin_amdgcn_ballot_w64(num != num); __builtin_expect(left != 0, 0);) {  // uniform over the wave
      const int rr = __shfl(r, __builtin_ctzll(left), 64), rt = rr / R, rh = rr - rt * R, at = ctx + rt;
      int hop = step;
      asm volatile("" : "+s"(hop));                           // (or the division is made in front of the loop)
      const int tiles = last_tile - first_tile + 1, mine = (tiles + hop - 1) / hop * kDaWaves;
      float* own = Ml + kDaWaves * 8 * 2 + wave * kPlainRowLds;
      const PlainRow row = plain_row(
          a, table, g, a.q + ((int64_t)(row0 + rt) * a.heads + g * R + rh) * a.dim, sig ? a.score_bias[g * R + rh] : 0.0f, at,
          max(low_of(at), 0), mine * kDaKeys,
          [&](int i) {
            const int t = i / kDaKeys;
            return (first_tile + t / kDaWaves * hop + (int)blockIdx.z * kDaWaves + t % kDaWaves) * kDaKeys + i % kDaKeys;
          },
          own);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      own[lane] = row.o[0];
      own[lane + 64] = row.o[1];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (r == rr) {
        // Where only a value is infinite the row's other channels may be another wave's, which keeps what it has: its maximum stands,
        // which lags behind by kDaGrowth at most.  Where scores are, every channel is worked out again.
        if (row.m > m_all + kDaGrowth + 0.5f) m_all = row.m;
        m_use = sink ? fmaxf(m_all, sk) : m_all;
        m_use = m_use == -INFINITY ? 0.0f : m_use;
        const float f = da_exp(row.m - m_use);
        den = f * row.l;
        num = f * own[c];
      }
      left &= ~__builtin_amdgcn_ballot_w64(r == rr);
    }
    if (e0 + lane >= rows * a.vdim) continue;
    if (sink) den += da_exp(sk - m_use);
    if (partial != nullptr) {
      const int64_t rh = (int64_t)(row0 + tt) * a.heads + g * R + hh, all = total_rows * a.heads;
      if (c == 0) {
        partial[(blockIdx.z * all + rh) * 2] = m_all;
        partial[(blockIdx.z * all + rh) * 2 + 1] = den;
      }
      partial[gridDim.z * all * 2 + (blockIdx.z * all + rh) * a.vdim + c] = num;
      continue;
    }
    float v = sig ? num : num / den;
    const int64_t col = (int64_t)(g * R + hh) * a.vdim + c;
    if (a.gate != nullptr) v *= sigmoidf_(ld<bf16_t>(a.gate, (row0 + tt) * a.gate_stride + col));
    st<bf16_t>(a.out, (row0 + tt) * a.out_stride + col, v);
  }
}

// Joins the parts, in a fixed order: a workgroup per (row, head)
__global__ __launch_bounds__(128) void decode_attention_join_kernel(const PromptAttention a, const float* __restrict__ partial,
                                                                    int64_t total_rows, int parts) {
  const int64_t rh = blockIdx.x, all = total_rows * a.heads, t = rh / a.heads;
  const int hd = (int)(rh - t * a.heads);
  const float* po = partial + parts * all * 2;
  const float sk = a.sink_logit != nullptr ? a.sink_logit[hd] : 0.0f;
  float m_all = a.sink ? sk : -INFINITY;
  for (int z = 0; z < parts; ++z) m_all = fmaxf(m_all, partial[(z * all + rh) * 2]);
  for (int c = threadIdx.x; c < a.vdim; c += 128) {
    float den = a.sink ? da_exp(sk - m_all) : 0.0f, num = 0.0f;
    for (int z = 0; z < parts; ++z) {
      const float f = da_exp(partial[(z * all + rh) * 2] - m_all);
      den += f * partial[(z * all + rh) * 2 + 1];
      num += f * po[(z * all + rh) * a.vdim + c];
    }
    float v = a.score_bias != nullptr ? num : num / den;
    const int64_t col = (int64_t)hd * a.vdim + c;
    if (a.gate != nullptr) v *= sigmoidf_(ld<bf16_t>(a.gate, t * a.gate_stride + col));
    st<bf16_t>(a.out, t * a.out_stride + col, v);
  }
}

template <int NB, int NS>
int launch_decode_attention(const PromptAttention& a, int64_t rows, int parts, float* workspace, hipStream_t stream) {
  static_assert(da_lds_bytes(NB) <= 80 * 1024, "two workgroups fit a compute unit");
  static_assert(kDecodeRows * 32 * NB * 4 <= kDaKeys * da_vstride(NB), "the outputs take the place of the staged values");
  auto kernel = decode_attention_kernel<NB, NS>;
  if (da_lds_bytes(NB) > 64 * 1024)
    SW_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     da_lds_bytes(NB)));
  hipLaunchKernelGGL(kernel, dim3((unsigned)a.num_seqs, (unsigned)a.kv_heads, (unsigned)parts), dim3(64 * kDaWaves),
                     da_lds_bytes(NB), stream, a, parts > 1 ? workspace : (float*)nullptr, rows);
  SW_CHECK_LAUNCH();
  if (parts > 1) {
    hipLaunchKernelGGL(decode_attention_join_kernel, dim3((unsigned)(rows * a.heads)), dim3(128), 0, stream, a, workspace, rows,
                       parts);
    SW_CHECK_LAUNCH();
  }
  return SW_OK;
}

int launch_decode_attention(const PromptAttention& a, int64_t rows, int max_query_len, float* workspace, hipStream_t stream) {
  const int parts = workspace == nullptr ? 1
                                         : decode_attention_parts(a.num_seqs, max_query_len, a.heads, a.kv_heads, a.page_size,
                                                                  a.table_width, a.window, a.chunk);
  const bool two = max_query_len * (a.heads / a.kv_heads) > 4;
#define SWM_DA_CASE(N)                                                                                                       \
  case N:                                                                                                                    \
    return two ? launch_decode_attention<N, 2>(a, rows, parts, workspace, stream)                                             \
               : launch_decode_attention<N, 1>(a, rows, parts, workspace, stream);
  switch ((std::max(a.dim, a.vdim) + 31) / 32) {
    SWM_DA_CASE(1)
    SWM_DA_CASE(2)
    SWM_DA_CASE(3)
    default: SWM_DA_CASE(4)
  }
#undef SWM_DA_CASE
}

}  // namespace swm
