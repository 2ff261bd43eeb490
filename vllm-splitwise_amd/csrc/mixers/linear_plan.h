// Which way the sequences of a linear-attention step go, and the sizes of the walk's launches and scratch.  Host code, no HIP
// headers.
#pragma once

#include <stdint.h>

namespace swm {

constexpr int kLwChunk = 32;

// Sequences of at most `at_most` tokens go through the kernels of decode steps (gla.hip, lightning.hip: a workgroup takes the whole
// run of a sequence and a head), longer ones through the walk.  -> at_most: 0: the walk takes all, max_query_len: the decode
// kernels do.  (us here / there, with norm and gate, the host's 30 a call included: 1 x 16 heads of 128, 16 tokens 32 / 34, 31 tokens
// 37 / 34, 64 tokens 63 / 34, 1000 tokens 921 / 75)
inline int linear_at_most(bool per_channel, int64_t rows, int num_seqs, int max_query_len, int heads, int dim, int vdim) {
  return max_query_len <= 16 ? max_query_len : 0;
}

// A walk's sizes.  Few runs leave most of the GPU idle, and a long run's chunks are then worth cutting: into segments whose own
// ends are worked out side by side, from nothing, and joined into the states that each segment truly starts from (one run of
// 16000 tokens, 4 heads of 128: 867 us in one piece, 8 segments: see linear_walk.hip).  As many as still leave every workgroup a
// compute unit, of at least 16 chunks.
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

}  // namespace swm
