// Host-side description of one compiled GEMM kernel instance ("algo") and the
// per-(epilogue, dtype) tables the C ABI dispatches through.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device.hpp"
#include "gemm_kernel.hpp"

namespace aitamd {

enum DType : int { kF16 = 0, kBF16 = 1, kNumDTypes = 2 };

struct GemmAlgo {
  const char* name;  // e.g. "gemm_rcr_f16_256x256x64_w2x2_v8"
  int bm, bn, bk;
  int threads;
  int kvec;
  int lds_bytes;
  int wgs_per_cu;  // workgroups of this instance one CU holds at once
  int direct_lds;  // 0: register-staged slabs, 1: direct-to-LDS ring, 2: persistent direct-to-LDS ring, 4: 1 + split-K, 8: few rows, 16: four waves
  int layouts;     // bit L set: a kernel for operand layout L exists (0 rcr, 1 rrr, 2 ccr, 3 crr)
  hipError_t (*launch)(const GemmParams& p, hipStream_t stream);
  // bytes of scratch memory (GemmParams::ws) a launch on this problem needs; null for instances that need none
  int64_t (*workspace_bytes)(const GemmParams& p);
  // what the instance choice reckons with, in us (see gemm_tiles.inc)
  struct {
    float start, mult, fetch, alone, tile;
  } cost;
};

struct GemmAlgoTable {
  const GemmAlgo* algos;
  int count;
  int residuals;  // operands of the result's size that the epilogue reads
};

// What the four-wave kernels store with their one epilogue: plain rows of whole 8-column pieces through buffer accesses.
inline bool four_waves_store(const GemmParams& p) {
  auto dwords = [](const void* v) { return (reinterpret_cast<uintptr_t>(v) & 3) == 0; };
  bool ok = p.perm_on == 0 && p.layout == 0 && (p.N & 7) == 0 && (p.ldc & 1) == 0 && (p.sc & 1) == 0 && (p.sc_outer & 1) == 0 &&
      dwords(p.c) && 256 * p.ldc * 2 < 0x7fffffffll;
  if (p.d0 != nullptr) ok = ok && (p.ldd & 1) == 0 && (p.sd & 1) == 0 && dwords(p.d0) && dwords(p.d1) && 256 * p.ldd * 2 < 0x7fffffffll;
  return ok;
}
// ... and multiply: K of three slab pairs at least
inline bool four_waves_multiply(int kvec, int64_t K) { return (kvec == 8 ? K : (K & ~7ll)) > 128; }

// What a split-K launch pays for sharing its tiles between s workgroups each, in us: three trips to memory (store, count,
// load), s workgroups that count and load, and the partial tiles' bytes.  Fitted, as are the slab times below,
// on 558 problems (M 21 to 1024, N 256 to 3072, K 512 to 8192) with every number of splits.
inline double split_k_exchange_us(int64_t tiles, int64_t s, int64_t tile_elems) {
  const double megabytes = (double)(tiles * s * tile_elems) * 4e-6;
  return tile_elems >= 128 * 128 ? 2.04 + 0.64 * (double)s + 0.34 * megabytes : 0.95 + 0.23 * (double)s + 0.48 * megabytes;
}

// Workgroups per tile of a split-K launch (the launcher and the instance choice share the rule): of the numbers from two
// up to about one workgroup per CU, with at least two K-slabs each, at most 16, the one that gives the least time for a
// workgroup's slabs and the exchange; 1 (no splitting, nothing written to the scratch memory) for grids that fill half
// the device anyway.  (The 32-deep slabs of 128 x 128 take as many as fill the CUs, a third more time than the best number: an
// instance that is never ahead of the others, for those who name it.)  Whether to split at all is the choice of the instance.  1.5 % (64 x 64 tiles) and 2.0 %
// (128 x 128) above the best number in the geometric mean; as many as fill the CUs, the rule before, 8 % and 21 %:
// 21 x 512 x 2048 11.5 us with 16, 7.1 with 4; 200 x 2304 x 768 in 128 x 128 tiles 17.4 with 6, 13.1 with 2.
// (128 x 128: measured on eight waves, the 0.395 us of a slab too.  On sixteen, which came after and take 0.96 to 1.03 times the
// time with the numbers of this rule, other numbers were not timed again.)
inline int split_k_rule(int64_t tiles, int64_t k_tiles, int bk, int64_t tile_elems, int cus) {
  if (tiles <= 0) return 1;
  if (bk < 64) {
    int64_t s = cus / tiles;
    if (s > k_tiles / 2) s = k_tiles / 2;
    if (s > 16) s = 16;
    return (int)(s < 1 ? 1 : s);
  }
  const double slab_us = (tile_elems >= 128 * 128 ? 0.395 : 0.226) * bk / 64;
  int best = 1;
  double best_us = 0;
  for (int64_t s = 2; s <= 16 && s * tiles <= cus && 2 * s <= k_tiles; ++s) {
    const double us = slab_us * (double)((k_tiles + s - 1) / s) + split_k_exchange_us(tiles, s, tile_elems);
    if (best == 1 || us < best_us) {
      best = (int)s;
      best_us = us;
    }
  }
  return best;
}

// Defined once per (epilogue, dtype) translation unit; nullptr table when that
// combination is not compiled in.
GemmAlgoTable gemm_table(int epilogue, int dtype);

}  // namespace aitamd
