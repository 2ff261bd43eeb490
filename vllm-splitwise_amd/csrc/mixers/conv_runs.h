// How the short convolution's workgroups share the rows of a step out (norm_conv.hip).  Host and device code, no HIP headers.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define SWM_HD __host__ __device__ inline
#else
#define SWM_HD inline
#endif

namespace swm {

enum ConvRows {
  kRowsElsewhere,  // rows t .. next - 1 belong to the workgroup of their sequence's first row
  kRowsInOrder,    // rows t .. next - 1 of one sequence, in order
  kRowAlone        // row t lies outside the sequence that its owner entry names: a row by itself, no state is touched
};
struct ConvPiece {
  ConvRows what;
  int64_t next;
};

// The piece that begins at row t of a workgroup whose run ends before row `end`; row t's sequence brings the rows
// [first, stop).  A sequence's first `keep` rows read the carried inputs and all belong to the workgroup of its first row, also
// those beyond the end of its run.  next > t whatever the arguments: a walk from piece to piece ends.
SWM_HD ConvPiece conv_piece(int64_t t, int64_t end, int64_t first, int64_t stop, int keep) {
  if (t < first || t >= stop) return {kRowAlone, t + 1};
  if (t > first && t < first + keep) return {kRowsElsewhere, first + keep < stop ? first + keep : stop};
  int64_t upto = end;
  if (t == first && first + keep > end) upto = first + keep;
  return {kRowsInOrder, upto < stop ? upto : stop};
}

}  // namespace swm
