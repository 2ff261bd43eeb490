// Waves of paged attention's vector kernel (paged_attention.cuh).  Host code, no HIP headers.
#pragma once

#include <stdint.h>

namespace sw {

// Launches of up to this many workgroups have 8 waves each, not 4: a workgroup's chain is half as long where the GPU has room for the waves
// (us, 4 / 8 waves, the write of the new tokens included: 32 heads of 128, 2 x 700 tokens 15.8 / 13.0, 8 x 700 24.2 / 20.3, 8 x 2000 62.3 / 55.5).  Twice
// as many where a token is 128 bytes of a head's keys (fp8 of 128, 16 bits of 64): 40 heads of 128, fp8, 8 x 1300 29.7 / 24.8, 8 x 1800
// 50.2 / 38.3, but 32 of 128, bf16, 10 x 2500 97.3 / 101.9.
// Contexts of up to 256 tokens are a walk of one step for 4 waves: 8 help there only where every workgroup writes all of the step's tokens
// (12 heads of 64, without a write 24 x 100 7.9 / 8.3, 40 x 40 8.0 / 8.3, with tokens looked up 40 x 10 4.9 / 5.5, 24 x 100 5.7 / 6.2; with all
// of them 40 heads of 128, 3 x 150 6.9 / 6.6, 4 x 150 8.6 / 8.2, 32 of 128, 2 x 40 5.27 / 5.39, 4 x 150 7.5 / 7.1).
constexpr int pa_wide_up_to(int key_bytes) { return key_bytes <= 128 ? 512 : 256; }
// longest: tokens that a context may have; writes_all: every workgroup writes all of the step's tokens into the cache first
constexpr bool pa_wide(int64_t workgroups, int key_bytes, int longest, bool writes_all) {
  return workgroups <= pa_wide_up_to(key_bytes) && (longest > 256 || writes_all);
}

// Whether every workgroup writes all of the step's tokens or looks up which of them it may read (PaWrite).  The lookup costs three barriers
// whatever it looks for, and takes a token for each sequence at most; writing all costs every workgroup each of the tokens.  us, looked up /
// all: 12 heads of 64, 4 x 800 tokens 8.64 / 8.60, 8 x 40 4.88 / 5.30, 16 x 40 5.00 / 6.06; 32 of 128, 2 x 400 8.90 / 8.76, 4 x 400 9.47 /
// 9.50, 6 x 400 11.1 / 11.5, 8 x 800 23.5 / 24.5, 16 x 40 8.2 / 13.0; 64 on 8, 4 x 150 6.97 / 6.72, 8 x 400 9.7 / 10.3.  Over 490 steps of 1 to
// 16 tokens this is 0.2 % behind the better of the two, at most 6 % in one (12 heads of 64, 4 x 150).
constexpr bool pa_writes_all(int tokens, int sequences) { return tokens <= 4 || tokens > sequences; }

}  // namespace sw
