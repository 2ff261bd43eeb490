// Which way the sequences of a linear-attention step go, and the sizes of the walk's launches and scratch.  Host code, no HIP
// headers.
#pragma once

#include <stdint.h>

namespace swm {

constexpr int kLwChunk = 32;

// A step with long runs is shared out between two ways: sequences of at most `at_most` tokens go through the kernels of decode
// steps (gla.hip, lightning.hip: a workgroup takes the whole run of a sequence and a head), longer ones through the walk.
// -> at_most: 0: the walk takes all, max_query_len: the decode kernels do.
// per_channel: decays per key channel (gla), else one per head, whose decode kernels are the cheaper ones.
// Measured (us a call of the rule alone; W: sequences x heads, of 128 x 128):
//   max_query_len <= 16: as decode steps, whatever W.
//   Sequences of about one length, decode kernels / walk.  With few the walk's chunks, side by side, win: W = 16, 100 tokens, per
//   channel 94 / 17.  With many the decode kernels fill the GPU by themselves and are spared the prologue's trip through memory:
//   per channel W = 256, 32 tokens 38 / 45, 64 tokens 75 / 55; W = 512, 64 tokens 95 / 95, 100 143 / 128, 150 218 / 159; W = 1024, 48
//   tokens 165 / 172, 100 282 / 278, 150 460 / 344.  Per head W = 256, 32 tokens 34 / 41, 64 58 / 51; W = 512, 64 tokens 76 / 86, 100
//   119 / 119, 200 202 / 176; W = 1024, 100 tokens 237 / 266, 150 308 / 328, 200 462 / 395.  (The lines were drawn for a walk of half
//   the speed: between them and the crossings above, at W = 512 and 1024 per head from 120 and 170 tokens on, calls take the slower way.)
//   Decoding sequences beside few long ones: all through the walk they are the dearest, 0.13 us a sequence and W; each its own way is the
//   cheapest from W = 160 on (us, all through the decode kernels / each its own way, 16 heads: per channel 60 sequences beside a portion of
//   24 tokens 55 / 42, 250 beside 24 154 / 129, per head 76 / 37, 268 / 123).
inline int linear_at_most(bool per_channel, int64_t rows, int num_seqs, int max_query_len, int heads, int dim, int vdim) {
  constexpr int kShort = 16;
  if (max_query_len <= kShort) return max_query_len;
  const int64_t w = (int64_t)num_seqs * heads;
  if (2 * rows >= (int64_t)max_query_len * num_seqs) {
    const int64_t most = per_channel ? w * dim / 512 - 16 : w * dim / 256 - 48, cap = per_channel ? 128 : 256;
    return max_query_len <= (most < kShort ? kShort : most > cap ? cap : most) ? max_query_len : 0;
  }
  const int64_t units = w * dim / 128;
  if (units > 160) return kShort;
  return max_query_len <= (units > 112 ? 24 : kShort) ? max_query_len : 0;
}

// Up to how many tokens a sequence that does not walk goes token by token with the state in whole rows (linear_step.hip; 0: none does)
// and not by chunks, whose kernels hold a state's columns (gla.hip, lightning.hip); max_query_len 0: not known.  Up to 5, where the
// per-channel rule's chunks go token by token too; beyond, its chunks round the state less often.  The state's error after 1600 tokens in
// portions, 4 heads of 128 x 128, token by token / by chunks: per channel 1.2e-6 / 1.2e-6 up to 5 tokens, chunks of 6 3.3e-7, of 13 3.0e-7; per
// head 7e-7 / 7e-7 for 1 token, 7e-7 / 4e-6 for 2, 8e-6 for 3, 3e-6 for 5 (every portion multiplies by the same rounded power of the decay).
// Measured, norm and gate included (us, by chunks / token by token), 16 heads of 128 x 128:
//   1 token each, 1 sequence: gla 13.1 / 8.0, lightning 29.0 / 9.7, retention 25.8 / 6.6; 61: 35.3 / 28.4, 74.1 / 30.4, 68.3 / 25.7;
//   4 tokens: 15.8 / 11.2, 29.2 / 12.3, 25.5 / 8.7; 61: 37.0 / 29.6, 70.1 / 29.2, 63.4 / 23.1.
// 8 heads of 256 x 256, 61 sequences, 1 token: 197 / 64, 186 / 65, 179 / 62.
// Where the rest of a step walks, runs of 6 tokens and more that do not are left to the chunks' kernels in a launch of their own, unless
// what is not a multiple of the longest run looks like most of them (20 of 12 tokens beside 300: 71 us without that launch, 74 with it).
// That looks at one long run: beside two of different length (512 and 400 tokens) decoding sequences go by chunks, as in steps whose
// longest run has 6 to 16 tokens.
inline int linear_step_tokens(int at_most, int64_t rows, int num_seqs, int max_query_len) {
  constexpr int kSteps = 5;
  if (max_query_len <= 0) return 0;
  const int longest = at_most < max_query_len ? at_most : max_query_len;
  if (longest <= kSteps) return longest;
  return at_most < max_query_len && rows % max_query_len <= kSteps * (int64_t)num_seqs ? kSteps : 0;
}

// A walk's sizes.  Few runs leave most of the GPU idle, and a long run's chunks are then worth cutting: into segments whose own
// ends are worked out side by side, from nothing, and joined into the states that each segment truly starts from (one run of
// 16000 tokens, 4 heads of 128: 448 us in one piece, 381 in 2, 218 in 4, 138 in 8; of 2000 tokens 71, 64, and 51 in 3).  As many as
// still leave every workgroup a compute unit, of at least 16 chunks.
struct LinearWalkPlan {
  int at_most, segment;                 // segment: tokens of a segment; 0: runs are not cut
  int64_t runs, chunks, items;          // upper bounds: runs that walk, their chunks, their segments
  int64_t floats;                       // of scratch
};
inline LinearWalkPlan linear_walk_plan(bool per_channel, int64_t rows, int num_seqs, int max_query_len, int heads, int dim, int vdim) {
  LinearWalkPlan p{linear_at_most(per_channel, rows, num_seqs, max_query_len, heads, dim, vdim), 0, 0, 0, 0, 0};
  if (p.at_most >= max_query_len) return p;
  const int64_t dp = (dim + 31) / 32 * 32, vblocks = (vdim + 15) / 16;
  p.runs = num_seqs;
  p.chunks = rows / kLwChunk + num_seqs;
  if (p.at_most > 0) {
    p.runs = rows / (p.at_most + 1) < p.runs ? rows / (p.at_most + 1) : p.runs;
    p.chunks = rows / kLwChunk + p.runs;
  }
  p.items = p.runs;
  // per chunk and head the scaled queries [32][dp], the scaled keys [dp][32], the decays [dp], the weights among its tokens [32][32]
  p.floats = p.chunks * heads * (65 * dp + 1024);
  const int64_t chunks = (max_query_len + kLwChunk - 1) / kLwChunk;
  const int64_t alike = (rows + max_query_len - 1) / max_query_len;     // runs about as long as the longest, at most about
  int64_t cuts = 256 / (alike * heads * vblocks);
  cuts = cuts < 16 ? cuts : 16;
  cuts = cuts < chunks / 16 ? cuts : chunks / 16;
  if (cuts >= 2) {
    p.segment = (int)((chunks + cuts - 1) / cuts) * kLwChunk;
    p.items = rows / p.segment + p.runs;
    p.floats += p.items * heads * (16 * vblocks * dp + dp);             // a segment's end state, its product of decays
  }
  return p;
}

// The walk's workgroups: one for each piece, head and 16 value channels, in eights of pieces and heads.
inline int64_t linear_walk_groups(const LinearWalkPlan& p, int heads, int vdim) {
  return (p.items * heads + 7) / 8 * 8 * ((vdim + 15) / 16);
}
// ... and how many of them are launched.  Beside decoding sequences the pieces are a far upper bound (a run for every 17 rows), and a
// workgroup that finds no piece still takes its turn in a compute unit that holds one of 8 waves at a time.  From 6 rounds of
// workgroups on two rounds of them go on to the next pieces instead, which costs a launch 1 - 2 us (their loop keeps more registers).
// us, one workgroup a piece / so; gla, heads of 128 unless stated.  5.8 rounds: 2 heads, 82 decoding sequences beside 10 portions,
// 49.1 / 48.7;  6.2: lightning, 16 of 64, 113 beside 10 67.0 / 65.8;  9: 32 heads, 61 beside 92 tokens 83.8 / 79.1;  29: 16 heads, 250
// beside 1000 tokens 237.6 / 177.7;  35: 32 heads, 96 beside 10 portions 202 / 172;  53: 8 of 256, 102 beside 4 550 / 458.
// One round: 79.1 -> 77.6 there, but lightning, 16 of 96, 21 beside 10 portions 85.5 -> 103.8: what a workgroup takes is settled then.
inline int64_t linear_walkers(const LinearWalkPlan& p, int heads, int dim, int vdim) {
  const int64_t groups = linear_walk_groups(p, heads, vdim), vblocks = (vdim + 15) / 16;
  const int64_t round = 256 * (dim <= 32 ? 4 : dim <= 96 ? 2 : 1);             // as many as the GPU holds at once, by their registers
  if (p.at_most == 0 || groups <= 6 * round) return groups;
  return (2 * round / vblocks + 7) / 8 * 8 * vblocks;
}

}  // namespace swm
