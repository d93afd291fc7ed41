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
//   kRows64:  two waves, 64 rows: short sequences, and those that leave the other half of 128 rows empty.
enum Form { kRows128 = 0, kRows256 = 1, kGroups = 2, kSmall = 3, kRows64 = 4 };

// The form for a problem, and whether causal query tiles go in pairs.
//
// What decides is how the workgroups of a form fill the chip: its iterations are the time of a grid that is not full,
// the work per CU that of a full one.  The lines lie where the forms' times cross over 780 problems (4 to 1000 sequences and
// heads, 16 to 8192 queries, keys as many or 77, head dims 32 to 160, 380 of them causal; each form timed in turn): a
// call takes 1.2 % more than in its best form in the geometric mean (5.6 % by the size of the grid alone, as before).
// Figures below: us, head dim 64 unless named, 256 CUs.
inline Form choose_form(int64_t B, int64_t M, int64_t N, int ks, int ot, bool causal, int cus, int32_t* paired) {
  const int64_t tiles128 = (M + 127) / 128;
  const int64_t t64 = (M + 63) / 64 * B, t128 = tiles128 * B, t256 = (M + 255) / 256 * B;
  // head dims up to 64: four workgroups of kRows128 on a CU, two of larger ones
  const bool narrow = ks <= 4 && ot <= 2, mid = !narrow && ks <= 6 && ot <= 3;
  *paired = 0;
  // Few queries: two groups halve the chain over the keys while all workgroups fit the chip at once (of kSmall one per CU at
  // head dims 128 and up, two below, three at 32).  64 x 1 x 4096 55 in one group, 32 in two; 554 x 21 x 1180 27.7 / 30.6.
  // Few keys give the second group nothing to share, three tiles of 32 too little: 48 x 28 x 28 at head dim 160 7.0 / 8.9.
  if (M <= 64) {
    const int64_t keys = causal && N > 64 ? 64 : N;  // (a causal tile stops behind its last row)
    const bool share = narrow || mid ? keys > 32 && (keys <= 64 || keys > 96) : keys > 192;
    return share && t64 <= cus * (ks <= 2 ? 3 : (narrow || mid ? 2 : 1)) ? kSmall : kRows64;  // 992 x 34^2: 6.6, 8.2 with 128 rows
  }
  // Few keys for more queries: 12 x 316 x 77 at head dim 128 8.4 in one group, 10.2 in two.  128 rows where they leave one
  // workgroup per CU (48 x 390 x 77 at head dim 32: 4.7, with 64 rows 5.3) and in large grids, which are wide or K and V are
  // read the less (272 x 3954 x 77 at head dim 40 59 / 67).
  if (N <= 96 || (ot > 4 && N <= 192))
    return t64 <= cus || (narrow && t128 > cus && (causal || t64 <= 8 * cus)) ? kRows64 : kRows128;
  // Grids that leave CUs idle: 64-row workgroups whose groups share the keys.  12 x 384^2 9.5 (128 rows, one group) / 8.6
  // (128, two) / 7.1 (64, two); 8 x 2048^2 at head dim 128 41 / 38 / 33.  A little beyond, while 128 rows still fill one
  // half of the chip: 12 x 2048^2 32.7 / 24 / 23.4; not at head dims 128 and up (60 x 275^2 11.4 / 12.4 / 19.2).
  if (t64 <= cus || ((narrow || mid) && N >= 256 && 16 * t64 <= 25 * cus)) return kSmall;
  if (causal) {
    // A workgroup's work grows with its rows' position.  Pairs of query tiles, the last with the first and so on, are all
    // the same length: best where they fill the chip in whole rounds (of one workgroup per CU with two groups, of two or
    // four without) and where there are enough tiles that an odd one in the middle is no matter.  Otherwise the longest
    // go first, and until the chip is full several times over the shortest chain counts: that of kSmall.
    // In order of length / pairs: 64 x 2048^2 59 / 50, 16 x 4096^2 at head dim 40 63 / 43, 36 x 3341^2 at 80 124 / 92;
    // 32 x 2237^2 45 / 53, and 39 with kSmall; 16 x 2346^2 at head dim 40 35 and 23; 24 x 1741^2 at 80 40 and 29.
    const bool pairable = B <= 65535 && (tiles128 % 2 == 0 || tiles128 >= 9);
    const int64_t pairs = (tiles128 + 1) / 2 * B;
    if (pairable && tiles128 >= 8 && 8 * pairs >= 7 * cus && pairs <= cus) {
      *paired = 1;
      return kGroups;
    }
    if (narrow) {
      const bool full = pairs >= 2 * cus;
      if (t64 <= 2 * cus || (!full && ((2 * t64 <= 9 * cus && M > 448) || M >= 1024))) return kSmall;
      // 64 rows while a pair of 128 would be a large part of the sequence: 276 x 508^2 31 / 27, 248 x 1781^2 144 / 160
      *paired = full && B <= 65535 && M >= 512;
      return M < 1536 ? kRows64 : kRows128;
    }
    if (mid ? t64 <= 2 * cus || (t64 <= 3 * cus && M >= 1024) : 4 * t64 <= 5 * cus && N >= 512) return kSmall;
    const int64_t rounds = (pairs + 2 * cus - 1) / (2 * cus);
    if (pairable && pairs >= cus && 10 * pairs >= 16 * cus * rounds) {  // (a last round four fifths full at least)
      *paired = 1;
      return kRows128;
    }
    if (t128 <= cus && N >= 512) return kGroups;
    return mid && M <= 512 ? kRows64 : kRows128;
  }
  if (t128 <= cus) return N >= 512 ? kGroups : kRows128;
  // Short sequences: smaller workgroups start and end more evenly.  816 x 135^2 20.5 (128 rows) / 17.8, 136 x 394^2 at
  // head dim 32 13.2 / 11.1; beyond, 768 x 384^2 of mixed lengths 41.2 / 41.6, 352 x 492^2 at head dim 40 33.0 / 35.2
  if (narrow && N <= (ks <= 2 ? 512 : 256)) return kRows64;
  // (head dim 32, where two groups' state is small: 64 x 1268^2 32.3 / 27.9)
  if (ks <= 2 && ot == 1 && N <= 4096 && t64 <= 8 * cus) return kSmall;
  // 64 rows per wave where K and V are read often enough to be the bound and the last round of the workgroups, two per
  // CU, is four fifths full: 16 x 8192^2 288, 312 with 32 rows; 64 x 2209^2 (1.1 rounds) 126 / 110; even at 62 x 4 x 1472^2
  // and at head dim 40
  const int64_t rounds = (t256 + 2 * cus - 1) / (2 * cus);
  if (ks == 4 && ot == 2 && M >= 2048 && 10 * t256 >= 16 * cus * rounds) return kRows256;
  return kRows128;
}

}  // namespace aitamd
