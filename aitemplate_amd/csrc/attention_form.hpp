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
// the work per CU that of a full one.  The lines lie where the forms' times cross over 8650 problems (4 to 1300 sequences and
// heads, 1 to 8192 queries, keys as many, 77 or any number, head dims 32 to 160, 4934 of them causal; each form timed in turn):
// a call takes 1.2 % more than in its best form in the geometric mean (5.2 % by the size of the grid alone).  A scheduler's luck
// with the last round is not in them: 4 % of the calls take 10 % more than in their best form.
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
  // workgroup per CU (48 x 390 x 77 at head dim 32: 4.7, with 64 rows 5.3) and in larger grids, which are wide or K and V are
  // read the less (168 x 748 x 77 12.0 / 14.2, 272 x 3954 x 77 at head dim 40 59 / 67), causal or not, unless they would leave
  // half of one in a few tiles empty (880 x 135 x 77 17.8 / 14.7).
  const bool half_empty = (M - 1) % 128 < 64;
  if (N <= 96 || (ot > 4 && N <= 192))
    return t64 <= cus || (narrow && t128 > cus && (2 * t64 <= 11 * cus || (half_empty && tiles128 <= 8))) ? kRows64 : kRows128;
  // Grids that leave CUs idle: 64-row workgroups whose groups share the keys.  12 x 384^2 9.5 (128 rows, one group) / 8.6
  // (128, two) / 7.1 (64, two); 8 x 2048^2 at head dim 128 41 / 38 / 33.  A little beyond, while 128 rows still fill one
  // half of the chip: 12 x 2048^2 32.7 / 24 / 23.4; not at head dims 128 and up (60 x 275^2 11.4 / 12.4 / 19.2).
  if (t64 <= cus || ((narrow || mid) && N >= 256 && 16 * t64 <= 25 * cus)) return kSmall;
  // (with half as many keys as queries most causal tiles are as long as one another: 32 x 3290 x 328 at head dim 40 17.1 in
  // 128 rows, 21.8 with kSmall)
  if (causal && 2 * N > M) {
    // A workgroup's work grows with its rows' position.  Pairs of query tiles, the last with the first and so on, are all
    // the same length: best where they fill the chip in whole rounds (of one workgroup per CU with two groups, of two or
    // four without) and where there are enough tiles that an odd one in the middle is no matter.  Otherwise the longest
    // go first, and until the chip is full several times over the shortest chain counts: that of kSmall.
    // In order of length / pairs: 64 x 2048^2 59 / 50, 16 x 4096^2 at head dim 40 63 / 43, 36 x 3341^2 at 80 124 / 92;
    // 32 x 2237^2 45 / 53, and 39 with kSmall; 24 x 1741^2 at 80 40 and 29.  Two groups, one pair per CU, from four fifths of
    // the CUs on (24 x 2161^2 at head dim 40 36 / 27; 16 x 2819^2 at 80 49, with kSmall 42), three quarters at head dims 128 and
    // up, where kSmall is slow (8 x 6164^2 132 / 107).
    const bool pairable = B <= 65535 && (tiles128 % 2 == 0 || tiles128 >= 9);
    const int64_t pairs = (tiles128 + 1) / 2 * B;
    if (pairable && tiles128 >= 8 && (narrow || mid ? 5 * pairs >= 4 * cus : 4 * pairs >= 3 * cus) && pairs <= cus) {
      *paired = 1;
      return kGroups;
    }
    if (narrow) {
      if (t64 <= 2 * cus) return kSmall;
      if (pairs < 2 * cus) {
        // 128 x 474^2 at head dim 40 12.4 in 128 rows, 12.9 in 64, 15.5 with kSmall, of which three fit a CU at head dim 32
        // (112 x 629^2 15.9 / 12.4); longer ones 96 x 1154^2 at 40 31.4 in pairs, 33.2; 100 x 1074^2 at 32 26.0, 23.7
        const bool small = M >= 900 ? ks <= 2 || t64 <= 6 * cus || M >= 4096 : M > 448 && 2 * t64 <= (ks <= 2 ? 9 : 7) * cus;
        if (small) return kSmall;
        *paired = M >= 900 && B <= 65535;
        return *paired ? kRows128 : kRows64;
      }
      // 64 rows while a pair of 128, or half a tile, would be a large part of the sequence: 276 x 508^2 31 / 27, 156 x 1143^2
      // (nine tiles of 128) 57 / 49, 200 x 702^2 35 / 31; 180 x 1274^2 66 / 74, 240 x 993^2 58 / 65
      *paired = B <= 65535 && M >= 512;
      return M < 512 || (M < 1536 && (tiles128 % 2 != 0 || half_empty)) ? kRows64 : kRows128;
    }
    // (at head dims 128 and up: 8 x 2563^2 at 160 71 in 128 rows, 58 in two groups of them, 50 with kSmall; 32 x 703^2 its 1.17)
    if (mid ? t64 <= 2 * cus || (t64 <= 3 * cus && M >= 1024) : N >= 512 && (4 * t64 <= 5 * cus || (M >= 2048 && 2 * t64 <= 3 * cus)))
      return kSmall;
    const int64_t rounds = (pairs + 2 * cus - 1) / (2 * cus);
    if (pairable && pairs >= cus && 10 * pairs >= 16 * cus * rounds) {  // (rounds four fifths full at least)
      *paired = 1;
      return kRows128;
    }
    if (t128 <= cus && N >= 512) return kGroups;
    return mid && M <= 512 ? kRows64 : kRows128;
  }
  if (t128 <= cus) return N >= 512 ? kGroups : kRows128;
  // Short sequences: 64 rows where 128 would leave half a tile empty, which starts and ends more evenly too, and while they are
  // few: 816 x 135^2 20.5 (128 rows) / 17.8; 768 x 200^2 at head dim 40 17.7 / 20.7, 768 x 256^2 27.0 / 29.4.  At head dim 32
  // where they are many (244 x 381^2 12.7 / 14.7, 384 x 392^2 the same).  Beyond, 768 x 384^2 of mixed lengths 41.2 / 41.6.
  if (narrow && N <= (ks <= 2 ? 512 : 256))
    return half_empty || (ks <= 2 ? t64 > 8 * cus : t64 <= 3 * cus) ? kRows64 : kRows128;
  // (head dim 32, where two groups' state is small: 64 x 1268^2 32.3 / 27.9)
  if (ks <= 2 && ot == 1 && N <= 4096 && t64 <= 8 * cus) return kSmall;
  // 64 rows per wave where K and V are read often enough to be the bound and the queries fill three quarters of the rounds of the
  // workgroups, two per CU: 16 x 8192^2 288, 312 with 32 rows; 64 x 4811^2 (0.78) 429 / 460, 60 x 3092^2 (0.71) 215 / 188
  const int64_t rounds = (t256 + 2 * cus - 1) / (2 * cus);
  if (ks == 4 && ot == 2 && M >= 2048 && M * B >= 384 * cus * rounds) return kRows256;
  return kRows128;
}

}  // namespace aitamd
