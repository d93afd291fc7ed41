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
  int32_t tiles_m, tiles_n;
  // Permuted store (kernels built with PERM; perm_on tells the launcher to pick them).  The row index splits as
  // m = (m0 * perm_m1 + m1) * perm_m2 + m2 and the column index as n = (n0 * perm_n1 + n1) * perm_n2 + n2,
  // and C[m, n] goes to element m0*sm0 + m1*sm1 + m2*sm2 + n0*sn0 + n1*sn1 + n2 of a contiguous buffer.
  // That covers the reference's 5-D output permutations
  // (python/aitemplate/backend/rocm/gemm/permute_common.py:20-130): "m2n3" has perm_m2 = 1, "m3n2" perm_n1 = 1.
  int32_t perm_on, perm_m1, perm_m2, perm_n1, perm_n2;
  int64_t perm_sm0, perm_sm1, perm_sm2, perm_sn0, perm_sn1;
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
  // Persistent kernels, one batch: when non-zero, XCD x owns the block of tiles_n / xcd_cols tile columns number
  // x % xcd_cols and tiles_m * xcd_cols / 8 tile rows number x / xcd_cols, and walks it row by row (see
  // map_tile_block).  Set by the launcher where the grid divides so and a block's B panels fit half an L2.
  int32_t xcd_cols;
  // Persistent kernels without the block mapping: tile rows per group of the grouped walk (0: eight).  An XCD's run
  // of consecutive tiles is walked group by group, column by column inside a group.
  int32_t group_m;
};

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
    const int m01 = m / p.perm_m2, m2 = m - m01 * p.perm_m2;
    const int m0 = m01 / p.perm_m1, m1 = m01 - m0 * p.perm_m1;
    const int n01 = n / p.perm_n2, n2 = n - n01 * p.perm_n2;
    const int n0 = n01 / p.perm_n1, n1 = n01 - n0 * p.perm_n1;
    return (m0 * p.perm_sm0 + m1 * p.perm_sm1 + m2 * p.perm_sm2) + (n0 * p.perm_sn0 + n1 * p.perm_sn1 + n2);
  }
}

}  // namespace aitamd
