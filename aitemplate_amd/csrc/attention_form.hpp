// Which form of the pipelined attention kernel (attention_pipe.hpp) a problem takes.  Host code only.
#pragma once

#include <stdint.h>

namespace aitamd {

// Work decompositions of the pipelined kernel.
//   kRows128: four waves of 32 query rows and tiles of 32 keys.  Head dims up to 64 fit four workgroups on a CU.
//   kRows256: four waves of 64 rows, which read every K and V fragment once for two matrix instructions; head dims of
//             one 64-wide instance only (the registers of larger ones leave a SIMD one wave, of smaller ones the
//             exponentials bound it and not the reads).
//   kGroups:  as kRows128 in eight waves, two groups on alternate halves of larger tiles.
//   kSmall:   two groups of two waves, 64 rows: four workgroups for every one of kGroups.
//   kRows64:  two waves, 64 rows: sequences that leave the other half of 128 rows empty.
enum Form { kRows128 = 0, kRows256 = 1, kGroups = 2, kSmall = 3, kRows64 = 4 };

// The form for a problem, and whether causal query tiles go in pairs (us below: head dim 64 unless named, one
// box, 256 CUs).
inline Form choose_form(int64_t B, int64_t M, int64_t N, int ks, int ot, bool causal, int cus, int32_t* paired) {
  const int64_t t64 = (M + 63) / 64, t128 = (M + 127) / 128, t256 = (M + 255) / 256;
  // Causal: a workgroup's work grows with its rows' position.  Pairs of query tiles, the last with the first and so on,
  // are all the same length: taken by one workgroup each where they fill the chip (two four-wave workgroups per CU or
  // one of two groups), and where there are enough tiles that an odd one in the middle is no matter.  Otherwise the
  // longest go first.  4 x 16 x 2048^2 59 / 50 (in order of length / pairs), 2 x 8 x 4096^2 at head dim 40 63 / 43.
  if (causal && B <= 65535 && (t128 % 2 == 0 || t128 >= 9)) {
    const int64_t pairs = (t128 + 1) / 2 * B;
    *paired = pairs >= 2 * cus || (t128 >= 8 && 4 * pairs >= 3 * cus && pairs <= cus);
    if (*paired) return pairs >= 2 * cus ? kRows128 : kGroups;
  }
  // Grids that leave CUs idle: 64-row workgroups whose groups share the keys; 128 rows while those do fill the chip.
  // 1 x 12 x 384^2 8.9 (128 rows, one group) / 8.5 (128, two) / 7.1 (64, two); 1 x 12 x 2048^2 31 / 24 / 24;
  // 1 x 8 x 2048^2 at head dim 128 41 / 38 / 33, at 512 workgroups of 64 rows (1 x 16 x 2000^2) 46 / 43 / 64.  Few
  // keys give the groups nothing to share: 6 x 12 x 316 x 77 at head dim 128 8.4 / 10.2 / 15.6.
  if (t64 * B <= cus || (16 * t64 * B <= 25 * cus && N >= 256)) return kSmall;
  if (M <= 64) return kRows64;  // 62 x 16 x 34^2: 6.6, 8.2 with 128 rows
  if (t128 * B <= cus && N >= 512) return kGroups;
  // 64 rows per wave where K and V are read often enough to be the bound: 1 x 16 x 8192^2 288, 312 with 32 rows; even
  // at 62 x 4 x 1472^2 and at head dim 40
  if (!causal && ks == 4 && ot == 2 && M >= 2048 && t256 * B >= 2 * cus) return kRows256;
  return kRows128;
}

}  // namespace aitamd
