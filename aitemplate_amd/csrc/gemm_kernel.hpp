// What the kernels of the RCR GEMM family share:  C[b][m][n] = epi( sum_k A[b][m][k] * B[b][n][k] ).
// A is row-major [M,K], B is row-major [N,K] (so both operands are K-contiguous), C is row-major [M,N] (other operand
// layouts: GemmParams::layout); fp16 or bf16 in/out, fp32 accumulate.
//
// The kernels replace the Composable Kernel device ops the reference instantiates for this
// family (python/aitemplate/utils/mk_ck_lib/gemm_operation.py:56-66, tile table
// python/aitemplate/utils/mk_ck_lib/generator.py:517-601,604-785,788-861).
#pragma once

#include "common.hpp"
#include "epilogue.hpp"

namespace aitamd {

struct GemmParams {
  const void* a;
  const void* b;
  void* c;
  const void* bias;  // [N]
  const void* d0;    // [M, ldd]
  const void* d1;    // [M, ldd]
  int32_t M, N, K;
  int32_t batch;
  int64_t lda, ldb, ldc, ldd;  // row pitches, in elements
  int64_t sa, sb, sc, sd;      // batch strides, in elements (0 broadcasts)
  // Set by the launcher (set_tiles): what a workgroup needs to find its tile.
  int32_t tiles_m, tiles_n;
  // Grouped walk: an XCD's run of consecutive tiles is walked in groups of 2^group_shift tile rows, column by column
  // inside a group.
  int32_t group_shift;
  // Persistent kernels, one batch: when not negative, XCD x owns the block of tiles_n >> xcd_shift tile columns number
  // x % 2^xcd_shift and of tiles_m >> (3 - xcd_shift) tile rows number x >> xcd_shift, and walks it row by row (see
  // map_tile).  Set where the grid divides so and a block's B panels fit half an L2.
  int32_t xcd_shift;
  // by tiles_m * tiles_n; by the tiles of a group (of a block's row, where the mapping is by blocks); by the rows of the
  // last group
  Divisor by_batch, by_group, by_last;
  // Permuted store (kernels built with PERM; perm_on tells the launcher to pick them).  The row index splits as
  // m = (m0 * perm_m1 + m1) * perm_m2 + m2 and the column index as n = (n0 * perm_n1 + n1) * perm_n2 + n2,
  // and C[m, n] goes to element m0*sm0 + m1*sm1 + m2*sm2 + n0*sn0 + n1*sn1 + n2 of a contiguous buffer.
  // That covers the reference's 5-D output permutations
  // (python/aitemplate/backend/rocm/gemm/permute_common.py:20-130): "m2n3" has perm_m2 = 1, "m3n2" perm_n1 = 1.
  int32_t perm_on, perm_m1, perm_m2, perm_n1, perm_n2;
  int64_t perm_sm0, perm_sm1, perm_sm2, perm_sn0, perm_sn1;
  Divisor by_perm_m1, by_perm_m2, by_perm_n1, by_perm_n2;  // (set by the launcher)
  // Non-zero: the output is written with streaming (non-temporal) stores.  Set by the launcher for outputs
  // too large to be still cached when a consumer runs; such stores do not push the operand tiles out of
  // the L2 and reach HBM at a higher rate (bmm_rcr 768x384x384x64: 4.1 -> 6.4 TB/s).
  int32_t nt_store;
  // Batched output whose batch index splits as b = b0 * batch_inner + b1 (0: plain batch stride sc): batch b
  // starts at element b0 * sc_outer + b1 * sc.  This is the [B/d1, d1, M, N] -> [B/d1, M, d1, N] store of
  // bmm_rcr_permute with batch_inner = d1, sc = N, sc_outer = M * d1 * N and ldc = d1 * N.
  int32_t batch_inner;
  int64_t sc_outer;
  // operand layout: 0 rcr (A [M, K], B [N, K]), 1 rrr (B [K, N]), 2 ccr (A [K, M]), 3 crr (both); lda / ldb
  // are the row pitches of the matrices as stored
  int32_t layout;
  // Scratch memory of the split-K instances (null for every other instance): arrival counters, then slots for
  // fp32 partial tiles; see gemm_kernel_dma.hpp.  The counters are zero before a launch and zero after it.
  void* ws;
  int64_t ws_bytes;
  int32_t split_k;  // number of workgroups that share a tile along K (set by the launcher of a split-K instance)
};

// The launcher's part of the walk over tiles of bm x bn.  xcd_shift: see GemmParams; -1 for the grouped walk.
inline void set_tiles(GemmParams& p, int bm, int bn, int group_shift, int xcd_shift) {
  p.tiles_m = (int32_t)(((int64_t)p.M + bm - 1) / bm);
  p.tiles_n = (int32_t)(((int64_t)p.N + bn - 1) / bn);
  p.group_shift = group_shift;
  p.xcd_shift = xcd_shift;
  const int last = p.tiles_m & ((1 << group_shift) - 1);
  p.by_batch = make_divisor((int64_t)p.tiles_m * p.tiles_n);
  p.by_group = make_divisor(xcd_shift >= 0 ? (int64_t)(p.tiles_n >> xcd_shift) : (int64_t)p.tiles_n << group_shift);
  p.by_last = make_divisor(last != 0 ? last : 1);
}

// Workgroup -> (batch entry, tile).  The hardware deals consecutive workgroup ids round-robin over the 8 XCDs; tiles that
// share an A row-panel or a B column-panel should land on the same XCD so the panel is fetched into one L2 only.  Two forms:
//  * grouped: every XCD gets a contiguous range of logical (batch, tile) ids, which are batch-major, so a range is a
//    run of whole batches (plus at most two partial ones at its ends): the tiles of one batch share its operands through
//    one L2 and fill its output rows together.  The tiles of a batch are walked in groups of tile rows, column by column.
//  * blocks (BLOCKS, where xcd_shift says so): XCD x works through its own block row by row, so the B panels of the
//    block's few columns are fetched into its L2 once and stay there for every row (the tiles that need an A panel
//    are adjacent in the walk and run at the same time).
template <bool BLOCKS = false>
AITAMD_DEVICE void map_tile(const GemmParams& p, int wg, int& b, int& tm, int& tn) {
  const int xcd = (int)((uint32_t)wg % kNumXcd), local = (int)((uint32_t)wg / kNumXcd);
  if (BLOCKS && p.xcd_shift >= 0) {
    const int cols = p.tiles_n >> p.xcd_shift, rows = p.tiles_m >> (3 - p.xcd_shift);
    const int r = quotient(local, p.by_group);
    b = 0;
    tm = (xcd >> p.xcd_shift) * rows + r;
    tn = (xcd & ((1 << p.xcd_shift) - 1)) * cols + (local - r * cols);
    return;
  }
  const int per_batch = p.tiles_m * p.tiles_n;
  const int total = per_batch * p.batch;
  const int q = (int)((uint32_t)total / kNumXcd), r = (int)((uint32_t)total % kNumXcd);
  const int flat = xcd * q + (xcd < r ? xcd : r) + local;
  b = p.batch > 1 ? quotient(flat, p.by_batch) : 0;
  const int id = flat - b * per_batch;
  const int first_m = quotient(id, p.by_group) << p.group_shift;
  const int in_group = id - first_m * p.tiles_n;
  // (the rows of a whole group are a power of two)
  const bool whole = p.tiles_m - first_m >= 1 << p.group_shift;
  const Divisor by_rows = {whole ? 1u : p.by_last.mul, whole ? (uint32_t)p.group_shift : p.by_last.shift};
  tn = quotient(in_group, by_rows);
  tm = first_m + (in_group - tn * (whole ? 1 << p.group_shift : p.tiles_m - first_m));
}

// All of these in registers here: left to itself the compiler fetches an argument when it gets to it, and a wait for one
// behind the arithmetic on another is a tenth of a microsecond each ahead of the first load of a tile.
AITAMD_DEVICE void fetch_arguments(const GemmParams& p) {
  asm volatile("" ::"s"(p.a), "s"(p.b), "s"(p.bias), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.batch), "s"(p.lda), "s"(p.ldb),
               "s"(p.tiles_m), "s"(p.tiles_n), "s"(p.by_group.mul), "s"(p.by_group.shift), "s"(p.by_last.mul), "s"(p.by_last.shift));
}

AITAMD_DEVICE int64_t out_batch_offset(const GemmParams& p, int batch) {
  if (p.batch_inner == 0) return (int64_t)batch * p.sc;
  const int b0 = batch / p.batch_inner;
  return b0 * p.sc_outer + (batch - b0 * p.batch_inner) * p.sc;
}

// Output store of 8 or 16 bytes at element `idx` of the buffer `rc` describes (base `base`).  The streaming
// form is a buffer store with the non-temporal bit; it is a different instruction from the plain store on
// purpose, so that the two branches cannot be folded into one plain store.
template <class T, class V>
AITAMD_DEVICE void store_out(T* base, int64_t idx, V v, bool streaming, __amdgpu_buffer_rsrc_t rc) {
  constexpr int kNonTemporal = 2;
  if (streaming) {
    if constexpr (sizeof(V) == 16)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rc, (uint32_t)(idx * 2), 0, kNonTemporal);
    else
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rc, (uint32_t)(idx * 2), 0, kNonTemporal);
  } else {
    store_vec(base + idx, v);
  }
}
// descriptor for store_out: the launcher sets nt_store only when one batch of the output spans < 2 GiB
constexpr uint32_t kStoreRecords = 0x7fffffffu;

// Element index of C[m, n] in the output buffer.  PERM is a template flag rather than a run-time test so
// that the plain kernels carry none of the index arithmetic (in the large tiles the extra live values
// cost registers the main loop needs).  The row and the column parts are separate so that a lane that
// keeps one of them fixed across stores evaluates it once.
template <bool PERM>
AITAMD_DEVICE int64_t out_index(const GemmParams& p, int m, int n) {
  if constexpr (!PERM) {
    return (int64_t)m * p.ldc + n;
  } else {
    const int m01 = quotient(m, p.by_perm_m2), m2 = m - m01 * p.perm_m2;
    const int m0 = quotient(m01, p.by_perm_m1), m1 = m01 - m0 * p.perm_m1;
    const int n01 = quotient(n, p.by_perm_n2), n2 = n - n01 * p.perm_n2;
    const int n0 = quotient(n01, p.by_perm_n1), n1 = n01 - n0 * p.perm_n1;
    return (m0 * p.perm_sm0 + m1 * p.perm_sm1 + m2 * p.perm_sm2) + (n0 * p.perm_sn0 + n1 * p.perm_sn1 + n2);
  }
}

}  // namespace aitamd
