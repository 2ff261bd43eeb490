// Which kernel an int4 GEMM goes to (quant_gemm.hip).  Host code, no HIP headers.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace sw {

// k across the waves of a workgroup, A from memory; tiles streamed through LDS, rows x columns; 128 x 256 tiles; the general 64-row tiles
enum class Int4Way { kAcrossWaves, k32x128, k64x64, k64x128, k128x128, k128x256, k64Rows };
inline bool int4_streamed(Int4Way w) { return w >= Int4Way::k32x128 && w <= Int4Way::k128x128; }

// The streamed tiles for a size, or kAcrossWaves / k128x256 where those are better.  A launch is one round of at most 256 workgroups where
// the tiles allow it; k is split as often as that leaves room for.  Measured at 46 matrices (1024 to 28672 k x 2048 to 57344 columns:
// 7B and 13B layers, whole and halved, and widths of 2048, 3072, 6144, 8192, 12288, 14336) and 9 to 256 rows, weights from memory, us:
inline Int4Way int4_tile(int64_t M, int64_t N, int64_t K) {
  auto tiles = [&](int rows, int cols) { return ((M + rows - 1) / rows) * ((N + cols - 1) / cols); };
  // what a workgroup goes through, in stages of 128 k
  auto stages = [&](int rows, int cols) {
    const int64_t t = tiles(rows, cols), splits = std::max<int64_t>(1, std::min(256 / t, K / 128));
    return (K / 128 + splits - 1) / splits * ((t + 255) / 256);
  };
  if (M <= 32) {
    // k across waves reads A from memory, once per 64 columns, and has nothing to set up: the streamed tile is ahead where a workgroup
    // has enough to go through, and the sooner the more rows (across waves / streamed: 5120 x 5120, 7 stages, 28 rows 11.3 / 12.1, 32
    // rows 12.0 / 12.1; 8192 x 10240, 22 stages, 12 rows 22.0 / 18.1, 16 rows 23.4 / 18.2).  Over 414 sizes 1.5 % slower on average than the
    // better of the two, at most 10 % slower than k across waves (20480 x 4096, 17 rows 17.7 / 19.4).
    return M > 8 && stages(32, 128) * M >= 320 ? Int4Way::k32x128 : Int4Way::kAcrossWaves;
  }
  auto named = [&]() {
    if (tiles(64, 64) <= 256) {
      // up to 64 rows always (128 columns instead: 13.2 -> 14.5 at 5120 x 5120, level at 13824 x 5120); with more rows where the
      // splits fill the chip or k is short (96 rows: 5120 k x 7680 18.2, 64 x 128 19.1; 6912 k x 5120 20.6 / 18.3)
      const int64_t t = tiles(64, 64), filled = 256 / t * t;
      if (M <= 64 || K <= 5120 || filled >= 224) return Int4Way::k64x64;
    }
    if (M <= 64) return Int4Way::k64x128;             // 5120 k x 27648 28.6, 64 x 64 in two rounds 38.0
    const int64_t t128 = tiles(128, 128);
    // 128 rows: 5120 k x 27648 43.0, 64 x 128 49.5; 5120 k x 15360 30.1 / 28.9, 4096 k x 12288 24.2 / 22.0
    if (M <= 128) return t128 > 128 ? Int4Way::k128x128 : Int4Way::k64x128;
    if (t128 > 256) return Int4Way::k128x256;
    // 192 rows: 6144 k x 8192 30.6 (192 tiles), 128 x 128 32.3; 13824 k x 5120 38.8 (120 tiles, 2 splits) / 44.2; 256 rows 60.9 (160 tiles) / 45.6
    const int64_t t = tiles(64, 128), filled = t <= 256 ? 256 / t * t : 0;
    return t <= 256 && (K <= 4096 || filled >= 180) ? Int4Way::k64x128 : Int4Way::k128x128;
  };
  const Int4Way way = named();
  // Above 64 rows a long walk is worth the wider tile in more splits: from 72 stages on (28672 x 8192, 112 stages, 65 rows 87.9 in tiles of
  // 64 x 64, 65.9 of 128 x 128; 256 rows 151.5 of 64 x 128, 125.3; 14336 x 8192, 256 rows 76.4 / 66.5; 20480 x 4096, 80 stages, 128 rows
  // 36.2 / 37.0; but 64 stages: 8192 x 10240, 160 rows 42.7 / 54.4, 8192 x 8192, 96 rows 26.5 / 28.6).
  if (M > 64 && tiles(128, 128) <= 256 &&
      ((way == Int4Way::k64x64 && stages(64, 64) >= 72) || (way == Int4Way::k64x128 && stages(64, 128) >= 72)))
    return Int4Way::k128x128;
  return way;
}

// on16: A lies on 16 bytes, which the streamed tiles ask for; room: it can be copied to such a place (worth it above 32 rows only)
inline Int4Way int4_way(int64_t M, int64_t N, int64_t K, int64_t group_size, bool on16, bool room) {
  if (K % 256 == 0) {
    const Int4Way way = int4_tile(M, N, K);
    if (int4_streamed(way) && (on16 || (room && M > 32))) return way;
    if (M > 128 && group_size % 64 == 0) return Int4Way::k128x256;
    if (M > 128 && group_size % 16 == 0) return Int4Way::k64Rows;
  }
  return Int4Way::kAcrossWaves;
}

}  // namespace sw
