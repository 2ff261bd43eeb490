// Prompt steps of the paged attention in capped_attention.hip over a bf16 cache, on the bf16 matrix cores without giving up
// fp32 scores and weights.
//
// What bounds it: matrix work.  The fp32 instructions (v_mfma_f32_32x32x2_f32) reach 154 TFLOP/s on this GPU, the bf16 ones
// nine times that.  Keys and values ARE bf16 numbers; queries and softmax weights are fp32 and are taken apart into three
// bf16 numbers each by truncation, x = h + m + l with 8 + 8 + 8 significant bits: the parts are exact, a bf16 x bf16 product
// is exact in fp32, so three bf16 products accumulated in fp32 are the fp32 product with its sums reordered -- at three
// times the work on units nine times as fast.  Except for an infinity in the cache, which a part that is zero turns into NaN: a row
// that comes out as NaN is worked out again in fp32 (plain_row), so the result is the fp32 product's there too.
//
// Tile: a group of 4 waves owns 4 x 32 query rows of one sequence and key/value head (row = token * R + head of the group, 32 / R
// tokens a wave) and walks the keys it sees in stages of 32 that the waves share through LDS: global -> registers two stages
// ahead, registers -> LDS one stage ahead, one barrier a stage.  Where walks are long a workgroup has TWO groups for the same rows,
// which take the stages in turn and join their sums at the end: under a causal mask the longest walk is twice the average one and the
// rest of the GPU would wait for it.  The two are half a stage apart, one at the products while the other is at the softmax; a SIMD
// has a wave of each.  What bounds a stage is the vector units (cap, softmax, taking weights apart: about 2300 cycles a wave), then the
// products (1536).
//   S^T = K Q^T : A = keys (row l % 32, 8 neighbouring coordinates per lane), B = the query parts, kept in registers;
//                 C element r of lane l: key 8 (r / 4) + 4 (l / 32) + r % 4, query l % 32.
//   O^T = V^T P^T: the score accumulator's layout is the B operand's, two runs of 4 keys per lane; A is read from the
//                 row-major value stage by the transposing ds_read_b64_tr_b16.
// The output is referred to a new running maximum only when some lane's has grown by more than 2^8 (weights are then below
// 2^8, sums stay in fp32 range, the factor cancels in the division).
// Workgroups are numbered latest tile of a sequence first: under a causal mask those have the longest walks.
//
// Measured, two prompts of 4324 tokens together, 16 query heads on 4 of size 128, capped scores and a gate: 989 us with the
// fp32 instructions (39 TFLOP/s), 177 us one group a workgroup, 159 us two; one prompt of 1607, 8 heads on 2, no cap: 88.7 and 69.2 us;
// two of 1296 behind 190 tokens each, 16 on 4: 95.7 and 74.8.  Error against 64 bits before the rounding to bf16: 1.3e-6 with the fp32
// instructions, 1.2e-6 here (without a cap 1.5 - 1.6e-7; 1.7 - 2.0e-7 with the small parts in a sum of their own).
#include "prompt_attention.cuh"

#include <algorithm>

namespace swm {

using pa_bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using pa_f32x16 = __attribute__((ext_vector_type(16))) float;
using pa_f32x4 = __attribute__((ext_vector_type(4))) float;
using pa_u32x4 = __attribute__((ext_vector_type(4))) uint32_t;
using pa_i16x4 = __attribute__((ext_vector_type(4))) short;
using pa_lds_i16x4 = __attribute__((address_space(3))) pa_i16x4*;

constexpr int kPaKeys = 32, kPaWaves = kPromptWaves;
constexpr float kLog2e = 1.4426950408889634f;

// one 16-byte fragment: 8 neighbouring bf16 numbers
union PaFrag {
  uint32_t w[4];
  pa_bf16x8 v;
};

// x = h + m + l, truncated to bf16 one after the other (exact); an infinity or NaN stays whole in h
__device__ __forceinline__ void split3(float x, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = __float_as_uint(x) & 0xffff0000u;
  const float r1 = (h & 0x7f800000u) == 0x7f800000u ? 0.0f : x - __uint_as_float(h);
  m = __float_as_uint(r1) & 0xffff0000u;
  l = __float_as_uint(r1 - __uint_as_float(m));
}
// the upper halves of two words, `lo` in the lower half
__device__ __forceinline__ uint32_t upper_halves(uint32_t hi, uint32_t lo) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); }

__host__ __device__ constexpr int pa_kstride(int nb) { return nb * 64 + 16; }                          // bytes per key row
__host__ __device__ constexpr int pa_vstride(int nb) { return (nb * 64 + 255) / 256 * 256 + 64; }      // bytes per value row
// a group's stages: two of keys, two of values; of two groups three of values, whose products come a turn later
__host__ __device__ constexpr int pa_lds_bytes(int nb, int groups) {
  return kPaKeys * (2 * pa_kstride(nb) + (groups > 1 ? 3 : 2) * pa_vstride(nb));
}

__host__ __device__ constexpr int pa_query_bytes(int nb) { return kPaWaves * 2 * 2 * nb * 1024; }         // two parts of the queries

// a wave's finished rows, or the row that it works out again
__host__ __device__ constexpr int pa_rows_bytes(int nb) {
  return 4 * (32 * (nb * 32 + 4) > kPlainRowLds ? 32 * (nb * 32 + 4) : kPlainRowLds);
}

// NB: blocks of 32 coordinates of the larger of key and value size.
// GROUPS: of 4 waves, which take the stages in turn, each with LDS buffers of its own; two of them have their sums meet at the end.
template <int NB, int GROUPS>
__global__ __launch_bounds__(64 * kPaWaves * GROUPS, 2) void prompt_attention_kernel(const PromptAttention a) {
  constexpr int KS = 2 * NB, CPR = 4 * NB, CHUNKS = kPaKeys * CPR, THREADS = 64 * kPaWaves;
  constexpr int LOADS = (CHUNKS + THREADS - 1) / THREADS;
  constexpr int KSTRIDE = pa_kstride(NB), VSTRIDE = pa_vstride(NB), VBUFS = GROUPS > 1 ? 3 : 2;
  extern __shared__ __attribute__((aligned(16))) char pa_lds[];
  const int tid = threadIdx.x % THREADS, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / THREADS);
  char* k_img = pa_lds + group * pa_lds_bytes(NB, GROUPS);           // [2][32][KSTRIDE]
  char* v_img = k_img + 2 * kPaKeys * KSTRIDE;               // [2 or 3][32][VSTRIDE]
  const int qi = lane & 31, hl = lane >> 5;
  const int R = a.heads / a.kv_heads, g = blockIdx.x % a.kv_heads;

  // ---- this workgroup's tile: sequences from the last, each one's tiles from its latest
  const int per_wg = kPaWaves * a.tpt;
  int tile = blockIdx.x / a.kv_heads, seq = -1, tok0 = 0, ntok = 0;
  for (int s = a.num_seqs - 1; s >= 0; --s) {
    const int n = a.q_start[s + 1] - a.q_start[s], tiles = (n + per_wg - 1) / per_wg;
    if (tile < tiles) {
      seq = s;
      tok0 = (tiles - 1 - tile) * per_wg;
      ntok = min(per_wg, n - tok0);
      break;
    }
    tile -= tiles;
  }
  if (seq < 0) return;                                       // the whole workgroup
  const int ctx = a.ctx_len[seq];
  const int32_t* table = a.block_tables + (int64_t)seq * a.table_width;
  // this wave's rows; a wave without tokens stages keys and meets barriers
  const int wtok = wave * a.tpt, nw = max(0, min(a.tpt, ntok - wtok));
  const int64_t row0 = (int64_t)a.q_start[seq] + tok0 + wtok;
  const int wfirst = ctx + tok0 + wtok, wlast = wfirst + nw - 1;
  const int tt = qi / R, hh = qi - tt * R;
  const bool row_ok = tt < nw;
  // rows without a token behave like the wave's last token and are never stored
  const int pos_q = wfirst + min(tt, max(nw - 1, 0));
  const int low_q = a.chunk > 0 ? pos_q / a.chunk * a.chunk : a.window > 0 ? pos_q - a.window + 1 : 0;
  auto lowest_of = [&](int first) {
    return a.chunk > 0 ? first / a.chunk * a.chunk : a.window > 0 ? max(0, first - a.window + 1) : 0;
  };
  const int wlow = lowest_of(wfirst);                                              // the wave's first key
  const int wlow_last = a.chunk > 0 ? wlast / a.chunk * a.chunk : a.window > 0 ? wlast - a.window + 1 : 0;   // its last row's
  const int last_pos = ctx + tok0 + ntok - 1;
  const int s_lo = lowest_of(ctx + tok0) / kPaKeys, s_hi = last_pos / kPaKeys;     // stages

  // ---- the queries' parts, scaled; scores live in the log2 domain unless a cap is applied to them first
  const bool sig = a.score_bias != nullptr, capped = a.softcap > 0.0f;
  const float qscale = capped ? a.scale : a.scale * kLog2e;
  const float cap2 = a.softcap * kLog2e, cap_in = capped ? 2.0f * kLog2e / a.softcap : 0.0f;
  const float bias2 = sig ? a.score_bias[g * R + hh] * kLog2e : 0.0f;
  // Two groups keep the leading parts in registers, the others in LDS, which both read.
  PaFrag qh[KS], qm_own[GROUPS > 1 ? 1 : KS], ql_own[GROUPS > 1 ? 1 : KS];
  pa_bf16x8* q_img = reinterpret_cast<pa_bf16x8*>(pa_lds + 2 * pa_lds_bytes(NB, GROUPS)) + wave * (2 * KS * 64) + lane;         // [part][KS][lane]
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    float x[8];
    const int c = 16 * ks + 8 * hl;
    const bool ok = row_ok && c < a.dim;
    const float* p = a.q + (row0 + tt) * (int64_t)a.heads * a.dim + (int64_t)(g * R + hh) * a.dim + c;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float4 v = ok ? *reinterpret_cast<const float4*>(p + 4 * j) : make_float4(0.f, 0.f, 0.f, 0.f);
      x[4 * j] = v.x * qscale; x[4 * j + 1] = v.y * qscale; x[4 * j + 2] = v.z * qscale; x[4 * j + 3] = v.w * qscale;
    }
    PaFrag qm, ql;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t h0, m0, l0, h1, m1, l1;
      split3(x[2 * j], h0, m0, l0);
      split3(x[2 * j + 1], h1, m1, l1);
      qh[ks].w[j] = upper_halves(h1, h0);
      qm.w[j] = upper_halves(m1, m0);
      ql.w[j] = upper_halves(l1, l0);
    }
    if constexpr (GROUPS > 1) {
      if (group == 0) {
        q_img[ks * 64] = qm.v;
        q_img[(KS + ks) * 64] = ql.v;
      }
    } else {
      qm_own[ks] = qm;
      ql_own[ks] = ql;
    }
  }

  // ---- staging: this thread's 16-byte pieces of a stage (key row c / CPR, piece c % CPR)
  int page_of[LOADS];
  pa_u32x4 kreg[LOADS], vreg[LOADS];
  auto key_of = [&](int it, int stage) { return min(stage * kPaKeys + (it * THREADS + tid) / CPR, last_pos); };
  auto tfetch = [&](int stage) {                             // page numbers, a stage before the pieces that they address
    sw::static_for<LOADS>([&](auto IT) {
      constexpr int it = decltype(IT)::value;
      const int key = key_of(it, stage);
      page_of[it] = table[a.page_shift >= 0 ? key >> a.page_shift : key / a.page_size];
    });
  };
  // (a page's place in one product of 32 by 32 bits, a key's in the page in 32, which attention_way sees to: 64-bit products took a
  // seventh of the vector units' time)
  const uint32_t krow = 2 * (uint32_t)a.k_stride, vrow = 2 * (uint32_t)a.v_stride;
  const uint32_t kpage = krow * (uint32_t)a.page_size, vpage = vrow * (uint32_t)a.page_size;
  auto fetch = [&](int stage) {
    sw::static_for<LOADS>([&](auto IT) {
      constexpr int it = decltype(IT)::value;
      const int c = it * THREADS + tid, ch = c % CPR, key = key_of(it, stage);
      const uint32_t in = a.page_shift >= 0 ? key & (a.page_size - 1) : key % a.page_size, page = page_of[it];
      pa_u32x4 kv = {0u, 0u, 0u, 0u}, vv = {0u, 0u, 0u, 0u};
      if ((CHUNKS % THREADS == 0 || c < CHUNKS)) {
        if (ch * 8 < a.dim)
          kv = *reinterpret_cast<const pa_u32x4*>(reinterpret_cast<const char*>(a.key_cache + g * a.dim + ch * 8) + (uint64_t)page * kpage +
                                                  in * krow);
        if (ch * 8 < a.vdim)
          vv = *reinterpret_cast<const pa_u32x4*>(reinterpret_cast<const char*>(a.value_cache + g * a.vdim + ch * 8) +
                                                  (uint64_t)page * vpage + in * vrow);
      }
      kreg[it] = kv;
      vreg[it] = vv;
    });
  };
  auto commit = [&](int kbuf, int vbuf) {
    sw::static_for<LOADS>([&](auto IT) {
      constexpr int it = decltype(IT)::value;
      const int c = it * THREADS + tid, key = c / CPR, ch = c % CPR;
      if (CHUNKS % THREADS == 0 || c < CHUNKS) {
        *reinterpret_cast<pa_u32x4*>(k_img + (kbuf * kPaKeys + key) * KSTRIDE + ch * 16) = kreg[it];
        *reinterpret_cast<pa_u32x4*>(v_img + (vbuf * kPaKeys + key) * VSTRIDE + ch * 16) = vreg[it];
      }
    });
  };
  // (one v_permlane32_swap; a shuffle through LDS would wait for an LDS round trip in every stage)
  auto other_half = [&](float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(hl ? r[0] : r[1]);
  };

  pa_f32x16 o[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[b][r] = 0.0f;
  float m_run = sig ? 0.0f : -INFINITY, l_part = 0.0f;
  // transposing reads: lane 4 i + p of a group of 16 names value row i, channels 4 p .. 4 p + 3 of a 4 x 16 block; the
  // wave's four groups are channels 0 / 16 of keys 0 / 4
  const int tr_off = (4 * (lane >> 5) + ((lane & 15) >> 2)) * VSTRIDE + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  const int k_off = qi * KSTRIDE + hl * 16;

  // This group's stages: first, first + GROUPS, ..  With two groups the same loads go on behind the last one, from the last key's
  // place: the compiler counts what is in flight, and under a condition would wait for all of it.
  const int first = s_lo + group, turns = (s_hi - s_lo + GROUPS) / GROUPS;
  auto live = [&](int t) {                                   // this wave sees keys of the stage (wave-uniform)
    const int k0 = (first + GROUPS * t) * kPaKeys;
    return nw > 0 && t >= 0 && t < turns && k0 <= wlast && k0 + kPaKeys > wlow;
  };
  pa_f32x16 s;
  PaFrag ph[2], pm[2], pl[2];
  // ---- the weights of 16 keys in parts (two groups: at the end of the vector half; one: in front of their products, which takes
  //      fewer registers)
  auto take_apart = [&](int st) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // (no infinity to look out for: a weight is at most 2^8)
      const float x0 = s[8 * st + 2 * j], x1 = s[8 * st + 2 * j + 1];
      const uint32_t h0 = __float_as_uint(x0) & 0xffff0000u, h1 = __float_as_uint(x1) & 0xffff0000u;
      const float r0 = x0 - __uint_as_float(h0), r1 = x1 - __uint_as_float(h1);
      const uint32_t m0 = __float_as_uint(r0) & 0xffff0000u, m1 = __float_as_uint(r1) & 0xffff0000u;
      ph[st].w[j] = upper_halves(h1, h0);
      pm[st].w[j] = upper_halves(m1, m0);
      pl[st].w[j] = upper_halves(__float_as_uint(r1 - __uint_as_float(m1)), __float_as_uint(r0 - __uint_as_float(m0)));
    }
  };
  // ---- O^T += V^T P^T, 16 keys at a time; B element j of a lane is key 16 st + 8 (j / 4) + 4 hl + j % 4
  auto value_products = [&](int vbuf) {
    const char* vb = v_img + vbuf * kPaKeys * VSTRIDE + tr_off;
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      if constexpr (GROUPS == 1) take_apart(st);
      pa_bf16x8 vf[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const char* base = vb + 16 * st * VSTRIDE + b * 64;
        union { pa_i16x4 half[2]; pa_bf16x8 f; } u;
        u.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pa_lds_i16x4)(base));
        u.half[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pa_lds_i16x4)(base + 8 * VSTRIDE));
        vf[b] = u.f;
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) o[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[b], pl[st].v, o[b], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < NB; ++b) o[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[b], pm[st].v, o[b], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < NB; ++b) o[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[b], ph[st].v, o[b], 0, 0, 0);
    }
  };
  // ---- S^T = K Q^T: the small parts of all coordinates in one sum; the leading ones on top of it, or in a second where registers
  //      are enough (the first sum, read once, is not waited for)
  auto key_products = [&](int t) {
    const char* kb = k_img + (t & 1) * kPaKeys * KSTRIDE + k_off;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.0f;
    if constexpr (GROUPS > 1) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const pa_bf16x8 kf = *reinterpret_cast<const pa_bf16x8*>(kb + 32 * ks);
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, q_img[(KS + ks) * 64], s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, q_img[ks * 64], s, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const pa_bf16x8*>(kb + 32 * ks), qh[ks].v, s, 0, 0, 0);
    } else {
      pa_f32x16 s2;
#pragma unroll
      for (int r = 0; r < 16; ++r) s2[r] = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const pa_bf16x8 kf = *reinterpret_cast<const pa_bf16x8*>(kb + 32 * ks);
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qh[ks].v, s, 0, 0, 0);
        s2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, ql_own[ks].v, s2, 0, 0, 0);
        s2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qm_own[ks].v, s2, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] += s2[r];
    }
  };
  // ---- the next stage into LDS, the one behind it on its way
  auto stage_next = [&](int t, int vbuf) {
    if (GROUPS > 1 || t + 1 < turns) commit((t + 1) & 1, vbuf == VBUFS - 1 ? 0 : vbuf + 1);
    if (GROUPS > 1 || t + 2 < turns) fetch(first + GROUPS * (t + 2));
    if (GROUPS > 1 || t + 3 < turns) tfetch(first + GROUPS * (t + 3));
  };
  // ---- the vector half: cap, mask, running softmax and the weights' parts (this lane: query qi, keys (r, hl))
  auto vector_half = [&](int t) {
    const int k0 = (first + GROUPS * t) * kPaKeys;
    if (capped) {
#pragma unroll
      for (int r = 0; r < 16; ++r)                           // cap * tanh(s / cap) = cap (1 - 2 / (1 + e^(2 s / cap)))
        s[r] = cap2 - 2.0f * cap2 * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(s[r] * cap_in));
    }
    if (k0 + kPaKeys - 1 > wfirst || k0 < wlow_last) {       // wave-uniform: something to mask
      const int hi = pos_q - k0 - 4 * hl, lo = low_q - k0 - 4 * hl;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int j = 8 * (r / 4) + r % 4;
        s[r] = j <= hi && j >= lo ? s[r] : -INFINITY;
      }
    }
    if (sig) {
#pragma unroll
      for (int r = 0; r < 16; ++r)                           // a hidden key: 1 / (1 + e^inf) = 0
        s[r] = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-(s[r] + bias2)));
    } else {
      float tmax = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) tmax = fmaxf(tmax, s[r]);
      const float m_new = fmaxf(m_run, fmaxf(tmax, other_half(tmax)));
      if (__builtin_amdgcn_ballot_w64(m_new > m_run + 8.0f) != 0) {
        const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.0f : m_new));
        l_part *= alpha;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[b][r] *= alpha;
        m_run = m_new;
      }
      const float m_use = m_run == -INFINITY ? 0.0f : m_run;
      float sum0 = 0.0f, sum1 = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        s[r] = __builtin_amdgcn_exp2f(s[r] - m_use);
        s[r + 1] = __builtin_amdgcn_exp2f(s[r + 1] - m_use);
        sum0 += s[r];
        sum1 += s[r + 1];
      }
      l_part += sum0 + sum1;
    }
    if constexpr (GROUPS > 1) {
      take_apart(0);
      take_apart(1);
    }
  };
  // ---- the finished rows go out 8 neighbouring channels a lane: piece 64 u + lane of 32 rows x 4 NB pieces (sizes are multiples of 8);
  //      rows without a token: the last one's again
  const bool gated = a.gate != nullptr && nw > 0;
  uint4 gates[2 * NB];
  auto place = [&](int u, int& row, int& c, int64_t& at_row, int& col) {
    const int i = 64 * u + lane;
    row = i / (4 * NB);
    c = i % (4 * NB) * 8;
    const int t = row / R;
    at_row = row0 + min(t, nw - 1);
    col = (g * R + row - t * R) * a.vdim + min(c, a.vdim - 8);
    return t < nw && c < a.vdim;
  };
  auto fetch_gates = [&]() {                                 // all of them, when the walk is through
    if (!gated) return;
    if (a.gate_stride % 8 == 0 && reinterpret_cast<uintptr_t>(a.gate) % 16 == 0) {
#pragma unroll
      for (int u = 0; u < 2 * NB; ++u) {
        int row, c, col;
        int64_t at_row;
        place(u, row, c, at_row, col);
        gates[u] = *reinterpret_cast<const uint4*>(a.gate + at_row * a.gate_stride + col);
      }
    } else {
#pragma unroll
      for (int u = 0; u < 2 * NB; ++u) {
        int row, c, col;
        int64_t at_row;
        place(u, row, c, at_row, col);
        const uint16_t* p = a.gate + at_row * a.gate_stride + col;
        gates[u] = make_uint4(p[0] | p[1] << 16, p[2] | p[3] << 16, p[4] | p[5] << 16, p[6] | p[7] << 16);
      }
    }
  };
  tfetch(first);
  fetch(first);
  if (GROUPS > 1 || turns > 1) tfetch(first + GROUPS);
  commit(0, 0);
  if (GROUPS > 1 || turns > 1) fetch(first + GROUPS);
  if (GROUPS > 1 || turns > 2) tfetch(first + 2 * GROUPS);
  __syncthreads();
  // A barrier a turn.  Of two groups one begins with the products, the other with the softmax of the stage before, so that a SIMD's
  // two waves are at different units.
  int vbuf = 0;                                              // t % VBUFS
  auto before = [&](int v) { return v == 0 ? VBUFS - 1 : v - 1; };
  if constexpr (GROUPS == 1) {
#pragma unroll 1
    for (int t = 0; t < turns; ++t, vbuf = vbuf == VBUFS - 1 ? 0 : vbuf + 1) {
      stage_next(t, vbuf);
      if (live(t)) {
        key_products(t);
        vector_half(t);
        value_products(vbuf);
      }
      __syncthreads();
    }
    fetch_gates();
  } else {
    if (group == 0) {
#pragma unroll 1
      for (int t = 0; t < turns; ++t, vbuf = vbuf == VBUFS - 1 ? 0 : vbuf + 1) {
        if (live(t - 1)) value_products(before(vbuf));
        if (live(t)) key_products(t);
        stage_next(t, vbuf);
        if (live(t)) vector_half(t);
        __syncthreads();
      }
      fetch_gates();
      if (live(turns - 1)) value_products(before(vbuf));
    } else {
#pragma unroll 1
      for (int t = 0; t < turns; ++t, vbuf = vbuf == VBUFS - 1 ? 0 : vbuf + 1) {
        stage_next(t, vbuf);
        if (live(t - 1)) {
          vector_half(t - 1);
          value_products(before(vbuf));
        }
        if (live(t)) key_products(t);
        __syncthreads();
      }
      if (live(turns - 1)) {
        vector_half(turns - 1);
        value_products(before(vbuf));
      }
    }
    __syncthreads();
    // ---- the second group's sums, referred to the larger maximum, into the first's
    static_assert(kPaWaves * (NB * 4096 + 512) <= 2 * pa_lds_bytes(NB, GROUPS), "the stages' LDS holds the sums");
    pa_f32x4* sums = reinterpret_cast<pa_f32x4*>(pa_lds) + wave * (NB * 256 + 32) + lane;
    float* rest = reinterpret_cast<float*>(pa_lds) + wave * (NB * 1024 + 128) + NB * 1024 + lane;
    if (group == 1) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
          sums[(b * 4 + r4) * 64] = pa_f32x4{o[b][4 * r4], o[b][4 * r4 + 1], o[b][4 * r4 + 2], o[b][4 * r4 + 3]};
      rest[0] = m_run;
      rest[64] = l_part;
    }
    __syncthreads();
    if (group == 0) {
      const float m1 = rest[0], l1 = rest[64];
      float a0 = 1.0f, a1 = 1.0f;
      if (!sig) {
        const float m = fmaxf(m_run, m1), m_use = m == -INFINITY ? 0.0f : m;
        a0 = __builtin_amdgcn_exp2f(m_run - m_use);
        a1 = __builtin_amdgcn_exp2f(m1 - m_use);
        m_run = m;
      }
      l_part = l_part * a0 + l1 * a1;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const pa_f32x4 x = sums[(b * 4 + r4) * 64];
#pragma unroll
          for (int r = 0; r < 4; ++r) o[b][4 * r4 + r] = o[b][4 * r4 + r] * a0 + x[r] * a1;
        }
    }
    __syncthreads();
    if (group != 0) return;
  }
  // ---- a row that came out as NaN again, in plain fp32 (the stages are done with: LDS is free, a part of it for each wave)
  int odd = 0;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) odd |= o[b][r] != o[b][r];
  const uint64_t lanes = __builtin_amdgcn_ballot_w64(row_ok && odd != 0);
  for (uint32_t left = (uint32_t)lanes | (uint32_t)(lanes >> 32); left != 0; left &= left - 1) {      // uniform over the wave
    const int r = __builtin_ctz(left), rt = r / R, rh = r - rt * R;
    const int pos = wfirst + rt, low = max(a.chunk > 0 ? pos / a.chunk * a.chunk : a.window > 0 ? pos - a.window + 1 : 0, 0);
    float* own = reinterpret_cast<float*>(pa_lds + wave * pa_rows_bytes(NB));
    const PlainRow row = plain_row(a, table, g, a.q + ((row0 + rt) * a.heads + g * R + rh) * (int64_t)a.dim,
                                   sig ? a.score_bias[g * R + rh] : 0.0f, pos, low, pos - low + 1, [&](int i) { return low + i; },
                                   own);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    own[lane] = row.o[0];
    own[lane + 64] = row.o[1];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (qi == r) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int c = 0; c < 16; ++c) o[b][c] = own[32 * b + 8 * (c / 4) + 4 * hl + c % 4];
      m_run = row.m * kLog2e;
      l_part = hl == 0 ? row.l : 0.0f;
    }
  }
  if (nw == 0) return;                                       // the whole wave

  // ---- normalise, gate, store: this lane holds query qi, channels 32 b + 8 (r / 4) + 4 hl + r % 4.  Through LDS, so that a lane
  //      stores 8 neighbouring channels and a short loop does it: from the accumulators' places it was 18 KB of instructions, gone
  //      through once, with a wait for a gate in front of every store (one prompt of 40 tokens, 16 heads on 4 of 128: 17.0 -> 14.4 us,
  //      two of 200: 25.4 -> 23.0, one of 700: 44.4 -> 42.1, four of 1000: 93.8 -> 91.4).  2 us of what is left are the gates' sigmoids;
  //      by the hardware's 2^x and reciprocal they would be 2^-18 off at gates near -84 and 0 from -87.4 on
  const float l_run = l_part + other_half(l_part);
  float inv = 1.0f;
  if (!sig) {
    // the sink: one more term that carries no value, of score 0 or of the head's learned score
    const float sk = a.sink_logit != nullptr ? a.sink_logit[g * R + hh] * kLog2e : 0.0f;
    const float m_fin = a.sink ? fmaxf(m_run, sk) : m_run;
    const float fin = a.sink ? __builtin_amdgcn_exp2f(m_run - m_fin) : 1.0f;
    inv = fin / (l_run * fin + (a.sink ? __builtin_amdgcn_exp2f(sk - m_fin) : 0.0f));
  }
  constexpr int OROW = NB * 32 + 4;                          // floats: 8 rows' quads on distinct banks
  float* rows_lds = reinterpret_cast<float*>(pa_lds + wave * pa_rows_bytes(NB));
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4)
      *reinterpret_cast<pa_f32x4*>(rows_lds + qi * OROW + 32 * b + 8 * r4 + 4 * hl) =
          pa_f32x4{o[b][4 * r4] * inv, o[b][4 * r4 + 1] * inv, o[b][4 * r4 + 2] * inv, o[b][4 * r4 + 3] * inv};
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const bool whole = a.out_stride % 8 == 0 && reinterpret_cast<uintptr_t>(a.out) % 16 == 0;
#pragma unroll 1
  for (int half = 0; half < 2; ++half)
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      int row, c, col;
      int64_t at_row;
      const bool mine = place(half * NB + u, row, c, at_row, col);
      const pa_f32x4 x0 = *reinterpret_cast<const pa_f32x4*>(rows_lds + row * OROW + c);
      const pa_f32x4 x1 = *reinterpret_cast<const pa_f32x4*>(rows_lds + row * OROW + c + 4);
      float v[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
      if (gated) {
        const uint4 gw = half ? gates[NB + u] : gates[u];
        const uint32_t w[4] = {gw.x, gw.y, gw.z, gw.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[2 * j] *= sigmoidf_(__uint_as_float(w[j] << 16));
          v[2 * j + 1] *= sigmoidf_(__uint_as_float(w[j] & 0xffff0000u));
        }
      }
      if (!mine) continue;
      uint16_t* op = static_cast<uint16_t*>(a.out) + at_row * a.out_stride + col;
      if (whole) {
        st_vec<bf16_t, 8>(op, 0, v);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) st<bf16_t>(op, j, v[j]);
      }
    }
}

template <int NB, int GROUPS>
int launch_prompt_tiles_as(const PromptAttention& a, unsigned groups, hipStream_t stream) {
  constexpr int lds = std::max(GROUPS * pa_lds_bytes(NB, GROUPS) + (GROUPS > 1 ? pa_query_bytes(NB) : 0), kPaWaves * pa_rows_bytes(NB));
  if (lds > 64 * 1024)
    SW_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(prompt_attention_kernel<NB, GROUPS>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  hipLaunchKernelGGL((prompt_attention_kernel<NB, GROUPS>), dim3(groups), dim3(64 * kPaWaves * GROUPS), lds, stream, a);
  SW_CHECK_LAUNCH();
  return SW_OK;
}

template <int NB>
int launch_prompt_tiles(const PromptAttention& a, int64_t rows, int max_query_len, hipStream_t stream) {
  const int64_t groups = prompt_attention_workgroups(rows, a.num_seqs, a.heads, a.kv_heads);
  SW_CHECK_ARG(groups < (1ll << 31), "masked_attention: too many rows");
  return prompt_attention_groups(rows, a.num_seqs, max_query_len, a.heads, a.kv_heads, a.page_size, a.table_width, a.window, a.chunk) > 1
             ? launch_prompt_tiles_as<NB, 2>(a, (unsigned)groups, stream)
             : launch_prompt_tiles_as<NB, 1>(a, (unsigned)groups, stream);
}

int launch_prompt_attention(const PromptAttention& a, int64_t rows, int max_query_len, hipStream_t stream) {
  switch ((std::max(a.dim, a.vdim) + 31) / 32) {
    case 1: return launch_prompt_tiles<1>(a, rows, max_query_len, stream);
    case 2: return launch_prompt_tiles<2>(a, rows, max_query_len, stream);
    case 3: return launch_prompt_tiles<3>(a, rows, max_query_len, stream);
    default: return launch_prompt_tiles<4>(a, rows, max_query_len, stream);
  }
}

}  // namespace swm
