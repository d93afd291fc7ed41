// C ABI of the RCR GEMM family: instance tables, support checks, the shape
// heuristic and the launchers declared in include/aitemplate_amd_kernels.h.
#include <stdio.h>
#include <string.h>

#include <mutex>
#include <string>

#include "../../include/aitemplate_amd_kernels.h"
#include "errors.hpp"
#include "gemm_host.hpp"

namespace aitamd {

// One declaration per compiled (epilogue, dtype) pair; the list is generated by the Makefile into gemm_tables.inc
// as AITAMD_TABLE(epi, dt) lines.  The references are weak: in the shared library every table is linked in, but a
// model library that links the static archive gets only the tables its generated op functions name (each names
// the table it dispatches through), and this file must not drag the other ones in.
#define AITAMD_TABLE(E, D) extern "C" __attribute__((weak)) GemmAlgoTable aitamd_gemm_table_##E##_##D();
#include "gemm_tables.inc"
#undef AITAMD_TABLE

GemmAlgoTable gemm_table(int epilogue, int dtype) {
#define AITAMD_TABLE(E, D) \
  if (epilogue == E && dtype == D) return &aitamd_gemm_table_##E##_##D ? aitamd_gemm_table_##E##_##D() : GemmAlgoTable{nullptr, 0, 0};
#include "gemm_tables.inc"
#undef AITAMD_TABLE
  return {nullptr, 0, 0};
}

namespace {

// layout: 0 rcr, 1 rrr (B is [K, N]), 2 ccr (A is [K, M]), 3 crr (both)
bool algo_supported(const GemmAlgo& a, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int align_bytes,
                    int layout = 0) {
  if (layout < 0 || layout > 3 || !(a.layouts & (1 << layout))) return false;
  const bool a_t = (layout & 2) != 0, b_t = (layout & 1) != 0;
  const int kv = a.kvec;
  if (align_bytes < kv * 2) return false;
  // an operand that is K-contiguous is fetched in pieces of kv elements along K; a transposed one in
  // 16-byte pieces along its rows of M (or N) elements, which only constrains its row pitch
  // (the register-staged instances read it in 16-byte pieces too, but at any address: any pitch)
  // With a padded pitch and M (or N) not a multiple of 8 the last 16-byte piece of k-row K-1 would reach past the
  // end of the operand (and of its buffer descriptor), so the row length has to be whole pieces as well.
  const int tv = a.direct_lds ? 8 : 1;
  if (a_t ? (lda % tv != 0 || M % tv != 0 || lda < M) : (K % kv != 0 || lda % kv != 0)) return false;
  if (b_t ? (ldb % tv != 0 || N % tv != 0 || ldb < N) : (K % kv != 0 || ldb % kv != 0)) return false;
  // Per-tile byte offsets are 32-bit, with the top bit reserved for "out of range".
  if ((a_t ? K * lda : (int64_t)a.bm * lda) * 2 >= 0x7fffffffll) return false;
  if ((b_t ? K * ldb : (int64_t)(a.direct_lds == 16 ? 256 : a.bn) * ldb) * 2 >= 0x7fffffffll) return false;
  if (M > 0x7fffffffll || K > 0x3fffffffll) return false;
  // the persistent kernels write a tile when its last K-slab has been multiplied: they need one
  if ((a.direct_lds == 2 || (a.direct_lds == 16 && kv == 8)) && K < 1) return false;
  return true;
}

int ptr_align(const void* p) {
  const uintptr_t v = reinterpret_cast<uintptr_t>(p);
  if (v == 0) return 16;
  int a = 1;
  while (a < 16 && (v & a) == 0) a <<= 1;
  return a;
}

// workgroups per tile of a split-K instance on this problem (the launcher's rule, gemm_inst.hip)
int split_factor(const GemmAlgo& a, int64_t batch, int64_t M, int64_t N, int64_t K, int cus) {
  const int64_t tiles = ((M + a.bm - 1) / a.bm) * ((N + a.bn - 1) / a.bn) * (batch > 0 ? batch : 1);
  const int64_t k_tiles = ((a.kvec == 8 ? K : (K & ~7)) + a.bk - 1) / a.bk;
  return split_k_rule(tiles, k_tiles, a.bk, (int64_t)a.bm * a.bn, cus);
}

// The instance with the smallest estimate of run time, from the measured figures that gemm_tiles.inc gives for each.
// Work is dealt in rounds of (CUs x workgroups per CU) tiles.  A CU with n workgroups takes n times an instance's
// slab time for a slab of each, but no less than the slab takes a workgroup that is alone there (it is then waiting
// for memory); a tile adds its fill and its epilogue.  The time that memory takes for the operands and the result goes on
// beside that: the longer of the two counts, and three tenths of the shorter.  Over 2100 linear layers and batched
// products of halves (gemm_tiles.inc) the choice is 1.3 % slower than the best instance on average, at 104 of them more than
// 10 %; the differences between runs of a launch of a few us are a good part of that.
int heuristic(const GemmAlgoTable& t, int64_t batch, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
              int align_bytes, int layout = 0, bool has_workspace = false, bool plain_store = true) {
  int best = -1;
  double best_cost = 0;
  const int kNumCu = current_device_cus();  // what the launcher sizes grids and split factors with
  const int64_t batches = batch > 0 ? batch : 1;
  const double memory_us = 2.0 * (double)batches * (double)(M * K + N * K + M * N) / 5.5e6;
  for (int i = 0; i < t.count; ++i) {
    const GemmAlgo& a = t.algos[i];
    if (!algo_supported(a, M, N, K, lda, ldb, align_bytes, layout)) continue;
    // (the twins for dword-aligned rows, and those for rows at any element, are for what the others cannot take)
    if (a.kvec == 2 && (a.direct_lds & 21) != 0 && align_bytes >= 16 && K % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0) continue;
    if (a.kvec == 1 && a.direct_lds == 8 && align_bytes >= 4 && K % 2 == 0 && lda % 2 == 0 && ldb % 2 == 0) continue;
    if (a.direct_lds == 16 && !(plain_store && N % 8 == 0 && four_waves_multiply(a.kvec, K))) continue;
    const int64_t whole = ((M + a.bm - 1) / a.bm) * ((N + a.bn - 1) / a.bn) * batches;
    // 128 x 128 through registers on sixteen waves has a CU to itself, its twin on eight shares one with a second workgroup,
    // which goes on while the first waits for its residuals or gathers a transposed B.  Over 2000 problems of odd K and layouts
    // that only these take, eight waves to sixteen: 1.04 to 1.12 the time up to one tile per CU; beyond that 1.00 to 1.04, but
    // 0.82 to 0.95 with residuals and 0.8 to 0.86 with B [K, N] (0.98 with both operands transposed).
    if (a.direct_lds == 0 && a.threads == 1024 && a.bm == 128 && whole > kNumCu && (t.residuals > 0 || (layout & 1))) continue;
    int64_t slabs = ((a.kvec == 2 && a.direct_lds != 8 ? K & ~7ll : K) + a.bk - 1) / a.bk;
    int64_t tiles = whole;
    double cost = a.cost.start;
    if (a.direct_lds == 4) {
      // split-K: usable with scratch memory, and worth a table entry of its own only where it does split (it is
      // the plain instance otherwise).  Every workgroup multiplies K / s.
      const int s_k = split_factor(a, batch, M, N, K, kNumCu);
      if (!has_workspace || s_k <= 1 || layout != 0) continue;
      slabs = (slabs + s_k - 1) / s_k;
      cost += split_k_exchange_us(tiles, s_k, (int64_t)a.bm * a.bn);
      tiles *= s_k;
    }
    const int per_cu = a.wgs_per_cu > 0 ? a.wgs_per_cu : 1;
    const int64_t slots = (int64_t)kNumCu * per_cu;
    const int64_t rounds = (tiles + slots - 1) / slots;
    const int64_t last = tiles - (rounds - 1) * slots;
    const int64_t busiest = (last + kNumCu - 1) / kNumCu;  // workgroups on the busiest CU in the last round
    // a tile wider or taller than the whole problem fetches only the rows that exist
    const double live = (double)((M < a.bm ? M : a.bm) + (N < a.bn ? N : a.bn)) / (a.bm + a.bn);
    const double fetch = a.cost.fetch * live;
    const double slab = fetch > a.cost.mult ? fetch : a.cost.mult;
    auto round_us = [&](double n) {
      const double full = n * slab;
      return (double)slabs * (full > a.cost.alone ? full : a.cost.alone) + n * a.cost.tile;
    };
    // the persistent kernel splits the tiles of a last round that would leave half the CUs idle over two CUs each
    const double last_frac = a.direct_lds == 2 && rounds > 1 && 2 * last <= kNumCu ? 0.72 : 1.0;
    const double work = (double)(rounds - 1) * round_us(per_cu) + last_frac * round_us((double)busiest);
    cost += work > memory_us ? work + 0.3 * memory_us : memory_us + 0.3 * work;
    // (between near equals not the four-wave kernel, which has one wave per SIMD for an epilogue; the fits are of a bias alone)
    if (a.direct_lds == 16) cost *= 1.06;
    // 256 x 256 through registers has one workgroup per CU and two slabs on their way: with K-contiguous rows at any element and
    // up to eight slabs a tile is mostly its fill and its store.  Over 300 problems of odd K it takes 1.04 to 1.2 times the better
    // 128 x 128 form's time there (2 to 8 slabs, 128 to 1024 tiles; 0.80 to 0.93 with more slabs), which its figures, fitted over
    // all K and layouts, do not say; transposed operands come in whole rows: 0.86 to 1.0.
    // (more than four rounds of tiles: 0.97 to 1.04, by the figures)
    if (a.direct_lds == 0 && a.bm == 256 && layout == 0 && K <= 512 && whole <= 4 * kNumCu) cost *= 1.14;
    if (best < 0 || cost < best_cost) {
      best = i;
      best_cost = cost;
    }
  }
  return best;
}

// The heuristic's answer for a problem, kept per thread for the problems last seen: scoring every instance takes
// 1.7 us of host time, as long as launching a small kernel, and a program calls with few distinct problems.  A
// direct-mapped table: a problem that maps to an occupied entry takes its place.
struct HeuristicKey {
  const GemmAlgo* table;
  int64_t batch, M, N, K, lda, ldb;
  int32_t align_bytes, layout, has_workspace, plain_store, cus;
  bool operator==(const HeuristicKey& o) const {
    return table == o.table && batch == o.batch && M == o.M && N == o.N && K == o.K && lda == o.lda && ldb == o.ldb &&
        align_bytes == o.align_bytes && layout == o.layout && has_workspace == o.has_workspace && plain_store == o.plain_store && cus == o.cus;
  }
};
int remembered_heuristic(const GemmAlgoTable& t, int64_t batch, int64_t M, int64_t N, int64_t K, int64_t lda,
                         int64_t ldb, int align_bytes, int layout, bool has_workspace, bool plain_store) {
  constexpr int kEntries = 256;
  struct Entry {
    HeuristicKey key{};
    int algo = -1;
  };
  static thread_local Entry entries[kEntries];
  const HeuristicKey key{t.algos, batch, M, N, K, lda, ldb, align_bytes, layout, has_workspace ? 1 : 0, plain_store ? 1 : 0, current_device_cus()};
  uint64_t h = reinterpret_cast<uint64_t>(t.algos);
  for (int64_t v : {batch, M, N, K, lda, ldb, (int64_t)(align_bytes * 16 + layout * 4 + key.has_workspace * 2 + key.plain_store)})
    h = (h ^ (uint64_t)v) * 0x9e3779b97f4a7c15ull;
  Entry& e = entries[h >> 56];
  if (!(e.key == key)) {
    e.algo = heuristic(t, batch, M, N, K, lda, ldb, align_bytes, layout, has_workspace, plain_store);
    e.key = key;
  }
  return e.algo;
}

int run_gemm(int epilogue, int dtype, int algo, const GemmParams& p, hipStream_t stream) {
  const GemmAlgoTable t = gemm_table(epilogue, dtype);
  if (t.count == 0) return fail("aitamd_gemm: no kernels compiled for epilogue %d dtype %d", epilogue, dtype);
  if (p.M < 0 || p.N < 0 || p.K < 0 || p.batch < 0) return fail("aitamd_gemm: negative dimension");
  if (p.M == 0 || p.N == 0 || p.batch == 0) return 0;
  if (!p.a && p.K > 0) return fail("aitamd_gemm: A pointer is null");
  if (!p.b && p.K > 0) return fail("aitamd_gemm: B pointer is null");
  if (!p.c) return fail("aitamd_gemm: C pointer is null");
  const bool a_t = (p.layout & 2) != 0, b_t = (p.layout & 1) != 0;
  if (p.lda < (a_t ? p.M : p.K) || p.ldb < (b_t ? p.N : p.K) || p.ldc < p.N)
    return fail("aitamd_gemm: row pitch smaller than the row");
  int align = ptr_align(p.a);
  const int ab = ptr_align(p.b);
  if (ab < align) align = ab;
  // batch strides shift the base pointers: fold them into the alignment.
  for (int64_t s : {p.sa, p.sb}) {
    if (s == 0) continue;
    int a2 = 1;
    while (a2 < 16 && ((s * 2) & a2) == 0) a2 <<= 1;
    if (a2 < align) align = a2;
  }
  if (algo < 0) {
    const bool plain = four_waves_store(p);
    algo = remembered_heuristic(t, p.batch, p.M, p.N, p.K, p.lda, p.ldb, align, p.layout, p.ws != nullptr && p.perm_on == 0, plain);
    // (the heuristic prices split-K with the split it would get; a buffer too small for that falls back)
    if (algo >= 0 && t.algos[algo].workspace_bytes && t.algos[algo].workspace_bytes(p) > p.ws_bytes)
      algo = remembered_heuristic(t, p.batch, p.M, p.N, p.K, p.lda, p.ldb, align, p.layout, false, plain);
    if (algo < 0) return fail("aitamd_gemm: no instance supports M=%d N=%d K=%d", p.M, p.N, p.K);
  }
  if (algo >= t.count) return fail("aitamd_gemm: algo %d out of range (have %d)", algo, t.count);
  const GemmAlgo& a = t.algos[algo];
  if (!algo_supported(a, p.M, p.N, p.K, p.lda, p.ldb, align, p.layout))
    return fail("aitamd_gemm: instance %s does not support M=%d N=%d K=%d lda=%lld ldb=%lld align=%d layout=%d", a.name,
                p.M, p.N, p.K, (long long)p.lda, (long long)p.ldb, align, p.layout);
  if (a.workspace_bytes && p.ws != nullptr && (reinterpret_cast<uintptr_t>(p.ws) & 15))
    return fail("aitamd_gemm: the workspace must be 16-byte aligned");
  const hipError_t e = a.launch(p, stream);
  if (e != hipSuccess) return fail("aitamd_gemm: launch of %s failed: %s", a.name, hipGetErrorString(e));
  return 0;
}

}  // namespace
}  // namespace aitamd

using namespace aitamd;

extern "C" {

const char* aitamd_version(void) { return "aitemplate_amd 0.1 gfx950"; }

const char* aitamd_last_error(void) { return last_error().c_str(); }

int aitamd_gemm_num_algos(int epilogue, int dtype) { return gemm_table(epilogue, dtype).count; }

const char* aitamd_gemm_algo_name(int epilogue, int dtype, int algo) {
  const GemmAlgoTable t = gemm_table(epilogue, dtype);
  if (algo < 0 || algo >= t.count) return nullptr;
  return t.algos[algo].name;
}

int aitamd_gemm_find_algo(int epilogue, int dtype, const char* name) {
  if (!name) return -1;
  const GemmAlgoTable t = gemm_table(epilogue, dtype);
  for (int i = 0; i < t.count; ++i)
    if (strcmp(t.algos[i].name, name) == 0) return i;
  return -1;
}

int aitamd_gemm_algo_supported(int epilogue, int dtype, int algo, int64_t M, int64_t N, int64_t K, int64_t lda,
                               int64_t ldb, int align_bytes) {
  const GemmAlgoTable t = gemm_table(epilogue, dtype);
  if (algo < 0 || algo >= t.count) return 0;
  return algo_supported(t.algos[algo], M, N, K, lda, ldb, align_bytes) ? 1 : 0;
}

int aitamd_gemm_algo_supported_layout(int epilogue, int dtype, int layout, int algo, int64_t M, int64_t N, int64_t K,
                                      int64_t lda, int64_t ldb, int align_bytes) {
  const GemmAlgoTable t = gemm_table(epilogue, dtype);
  if (algo < 0 || algo >= t.count) return 0;
  // (the four-wave instances hand a permuted store on to a small tile: no candidates for one)
  if (layout == AITAMD_LAYOUT_RCR_PERMUTED && t.algos[algo].direct_lds == 16) return 0;
  return algo_supported(t.algos[algo], M, N, K, lda, ldb, align_bytes, layout == AITAMD_LAYOUT_RCR_PERMUTED ? 0 : layout) ? 1 : 0;
}

int aitamd_gemm_heuristic_algo_layout(int epilogue, int dtype, int layout, int64_t batch, int64_t M, int64_t N,
                                      int64_t K, int64_t lda, int64_t ldb, int align_bytes) {
  const GemmAlgoTable t = gemm_table(epilogue, dtype);
  if (t.count == 0) return -1;
  return heuristic(t, batch, M, N, K, lda, ldb, align_bytes, layout == AITAMD_LAYOUT_RCR_PERMUTED ? 0 : layout, false, layout != AITAMD_LAYOUT_RCR_PERMUTED);
}

int aitamd_gemm_heuristic_algo(int epilogue, int dtype, int64_t batch, int64_t M, int64_t N, int64_t K, int64_t lda,
                               int64_t ldb, int align_bytes) {
  const GemmAlgoTable t = gemm_table(epilogue, dtype);
  if (t.count == 0) return -1;
  return heuristic(t, batch, M, N, K, lda, ldb, align_bytes);
}

int64_t aitamd_gemm_workspace_bytes(int epilogue, int dtype, int algo, int64_t batch, int64_t M, int64_t N, int64_t K) {
  const GemmAlgoTable t = gemm_table(epilogue, dtype);
  if (algo < 0 || algo >= t.count || !t.algos[algo].workspace_bytes) return 0;
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0 || M > 0x7fffffffll || N > 0x7fffffffll || K > 0x7fffffffll) return 0;
  GemmParams p{};
  p.M = (int32_t)M;
  p.N = (int32_t)N;
  p.K = (int32_t)K;
  p.batch = (int32_t)batch;
  return t.algos[algo].workspace_bytes(p);
}

int aitamd_gemm_rcr(int epilogue, int dtype, int algo, const void* a, const void* b, const void* bias, const void* d0,
                    const void* d1, void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc,
                    int64_t ldd, void* stream) {
  return aitamd_gemm_rcr_ws(epilogue, dtype, algo, a, b, bias, d0, d1, c, M, N, K, lda, ldb, ldc, ldd, nullptr, 0, stream);
}

int aitamd_gemm_rcr_ws(int epilogue, int dtype, int algo, const void* a, const void* b, const void* bias,
                       const void* d0, const void* d1, void* c, int64_t M, int64_t N, int64_t K, int64_t lda,
                       int64_t ldb, int64_t ldc, int64_t ldd, void* workspace, int64_t workspace_bytes, void* stream) {
  if (epilogue < 0 || epilogue >= kNumEpilogues) return fail("aitamd_gemm_rcr: bad epilogue id %d", epilogue);
  if (M > 0x7fffffffll || N > 0x7fffffffll || K > 0x7fffffffll) return fail("aitamd_gemm_rcr: dimension too large");
  GemmParams p{};
  p.a = a;
  p.b = b;
  p.c = c;
  p.bias = bias;
  p.d0 = d0;
  p.d1 = d1;
  p.M = (int32_t)M;
  p.N = (int32_t)N;
  p.K = (int32_t)K;
  p.batch = 1;
  p.lda = lda;
  p.ldb = ldb;
  p.ldc = ldc;
  p.ldd = ldd;
  p.ws = workspace_bytes > 0 ? workspace : nullptr;
  p.ws_bytes = p.ws ? workspace_bytes : 0;
  if (M > 0 && N > 0) {
    const bool need_bias = epilogue != kEpiNone && epilogue != kEpiAdd;
    const bool need_d0 = epilogue == kEpiBiasAdd || epilogue == kEpiBiasAddAdd || epilogue == kEpiBiasAddRelu ||
        epilogue == kEpiBiasAddAddRelu || epilogue >= kEpiBiasMul;
    const bool need_d1 = epilogue == kEpiBiasAddAdd || epilogue == kEpiBiasAddAddRelu || epilogue == kEpiBiasMulAdd;
    if (need_bias && !bias) return fail("aitamd_gemm_rcr: epilogue %d needs a bias pointer", epilogue);
    if (need_d0 && !d0) return fail("aitamd_gemm_rcr: epilogue %d needs d0", epilogue);
    if (need_d1 && !d1) return fail("aitamd_gemm_rcr: epilogue %d needs d1", epilogue);
    if (need_d0 && ldd < N) return fail("aitamd_gemm_rcr: residual pitch smaller than N");
  }
  return run_gemm(epilogue, dtype, algo, p, reinterpret_cast<hipStream_t>(stream));
}

int aitamd_gemm_permute(int operands, int epilogue, int dtype, int algo, const void* a, const void* b,
                        const void* bias, void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                        int layout, int64_t g1, int64_t g2, int64_t g3, void* stream);

int aitamd_gemm_rcr_permute(int epilogue, int dtype, int algo, const void* a, const void* b, const void* bias, void* c,
                            int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int layout, int64_t g1,
                            int64_t g2, int64_t g3, void* stream) {
  return aitamd_gemm_permute(AITAMD_LAYOUT_RCR, epilogue, dtype, algo, a, b, bias, c, M, N, K, lda, ldb, layout, g1, g2,
                             g3, stream);
}

int aitamd_gemm_permute(int operands, int epilogue, int dtype, int algo, const void* a, const void* b,
                        const void* bias, void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                        int layout, int64_t g1, int64_t g2, int64_t g3, void* stream) {
  if (operands != AITAMD_LAYOUT_RCR && !(operands == AITAMD_LAYOUT_RRR && epilogue == kEpiBias))
    return fail("aitamd_gemm_permute: operand layout %d with epilogue %d has no permuted store", operands, epilogue);
  if (epilogue < 0 || epilogue >= kNumEpilogues) return fail("aitamd_gemm_rcr_permute: bad epilogue id %d", epilogue);
  if (epilogue != kEpiNone && epilogue != kEpiBias)
    return fail("aitamd_gemm_rcr_permute: only the plain and the bias epilogue have a permuted store, not %d", epilogue);
  if (M > 0x7fffffffll || N > 0x7fffffffll || K > 0x7fffffffll) return fail("aitamd_gemm_rcr_permute: dimension too large");
  if (M < 0 || N < 0 || g1 <= 0 || g2 <= 0 || g3 <= 0)
    return fail("aitamd_gemm_rcr_permute: bad sizes M=%lld N=%lld g=(%lld, %lld, %lld)", (long long)M, (long long)N,
                (long long)g1, (long long)g2, (long long)g3);
  GemmParams p{};
  p.perm_on = 1;
  p.layout = operands;
  if (layout == AITAMD_PERMUTE_M2N3) {
    // [M0, M1 = g1, N0 = g2, N1 = g3, N2] -> [N0, M0, N1, M1, N2]
    if (M % g1 != 0 || N % (g2 * g3) != 0)
      return fail("aitamd_gemm_rcr_permute: m2n3 needs g1 | M and g2*g3 | N (M=%lld N=%lld g=(%lld, %lld, %lld))",
                  (long long)M, (long long)N, (long long)g1, (long long)g2, (long long)g3);
    const int64_t M0 = M / g1, M1 = g1, N1 = g3, N2 = N / (g2 * g3);
    p.perm_m1 = (int32_t)M1;
    p.perm_m2 = 1;
    p.perm_n1 = (int32_t)N1;
    p.perm_n2 = (int32_t)N2;
    p.perm_sm0 = N1 * M1 * N2;
    p.perm_sm1 = N2;
    p.perm_sm2 = 0;
    p.perm_sn0 = M0 * N1 * M1 * N2;
    p.perm_sn1 = M1 * N2;
  } else if (layout == AITAMD_PERMUTE_M3N2) {
    // [M0, M1 = g1, M2 = g2, N0 = g3, N1] -> [M2, M0, N0, M1, N1]
    if (M % (g1 * g2) != 0 || N % g3 != 0)
      return fail("aitamd_gemm_rcr_permute: m3n2 needs g1*g2 | M and g3 | N (M=%lld N=%lld g=(%lld, %lld, %lld))",
                  (long long)M, (long long)N, (long long)g1, (long long)g2, (long long)g3);
    const int64_t M0 = M / (g1 * g2), M1 = g1, M2 = g2, N0 = g3, N1 = N / g3;
    p.perm_m1 = (int32_t)M1;
    p.perm_m2 = (int32_t)M2;
    p.perm_n1 = 1;
    p.perm_n2 = (int32_t)N1;
    p.perm_sm0 = N0 * M1 * N1;
    p.perm_sm1 = N1;
    p.perm_sm2 = M0 * N0 * M1 * N1;
    p.perm_sn0 = M1 * N1;
    p.perm_sn1 = 0;
  } else {
    return fail("aitamd_gemm_rcr_permute: layout %d is not implemented", layout);
  }
  p.a = a;
  p.b = b;
  p.c = c;
  p.bias = bias;
  p.M = (int32_t)M;
  p.N = (int32_t)N;
  p.K = (int32_t)K;
  p.batch = 1;
  p.lda = lda;
  p.ldb = ldb;
  p.ldc = N;
  p.ldd = N;
  if (M > 0 && N > 0 && epilogue != kEpiNone && !bias)
    return fail("aitamd_gemm_rcr_permute: epilogue %d needs a bias pointer", epilogue);
  return run_gemm(epilogue, dtype, algo, p, reinterpret_cast<hipStream_t>(stream));
}

int aitamd_bmm_rcr(int dtype, int algo, const void* a, const void* b, void* c, int64_t batch, int64_t M, int64_t N,
                   int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t stride_a, int64_t stride_b,
                   int64_t stride_c, void* stream) {
  if (M > 0x7fffffffll || N > 0x7fffffffll || K > 0x7fffffffll || batch > 0x7fffffffll)
    return fail("aitamd_bmm_rcr: dimension too large");
  GemmParams p{};
  p.a = a;
  p.b = b;
  p.c = c;
  p.M = (int32_t)M;
  p.N = (int32_t)N;
  p.K = (int32_t)K;
  p.batch = (int32_t)batch;
  p.lda = lda;
  p.ldb = ldb;
  p.ldc = ldc;
  p.ldd = ldc;
  p.sa = stride_a;
  p.sb = stride_b;
  p.sc = stride_c;
  return run_gemm(kEpiNone, dtype, algo, p, reinterpret_cast<hipStream_t>(stream));
}

int aitamd_bmm_rcr_permute(int dtype, int algo, const void* a, const void* b, void* c, int64_t batch, int64_t M,
                           int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t stride_a, int64_t stride_b,
                           int64_t d1, void* stream) {
  if (M > 0x7fffffffll || N > 0x7fffffffll || K > 0x7fffffffll || batch > 0x7fffffffll)
    return fail("aitamd_bmm_rcr_permute: dimension too large");
  if (d1 <= 0 || batch % d1 != 0)
    return fail("aitamd_bmm_rcr_permute: batch %lld is not a multiple of d1 = %lld", (long long)batch, (long long)d1);
  GemmParams p{};
  p.a = a;
  p.b = b;
  p.c = c;
  p.M = (int32_t)M;
  p.N = (int32_t)N;
  p.K = (int32_t)K;
  p.batch = (int32_t)batch;
  p.lda = lda;
  p.ldb = ldb;
  // [B/d1, d1, M, N] -> [B/d1, M, d1, N]
  p.ldc = d1 * N;
  p.ldd = p.ldc;
  p.sa = stride_a;
  p.sb = stride_b;
  p.sc = N;
  p.batch_inner = (int32_t)d1;
  p.sc_outer = M * d1 * N;
  return run_gemm(kEpiNone, dtype, algo, p, reinterpret_cast<hipStream_t>(stream));
}

int aitamd_bmm(int layout, int dtype, int algo, const void* a, const void* b, void* c, int64_t batch, int64_t M,
               int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t stride_a, int64_t stride_b,
               int64_t stride_c, int64_t d1, void* stream) {
  if (layout < AITAMD_LAYOUT_RCR || layout > AITAMD_LAYOUT_CRR) return fail("aitamd_bmm: unknown layout %d", layout);
  if (M > 0x7fffffffll || N > 0x7fffffffll || K > 0x7fffffffll || batch > 0x7fffffffll)
    return fail("aitamd_bmm: dimension too large");
  if (d1 < 0 || (d1 > 0 && batch % d1 != 0))
    return fail("aitamd_bmm: batch %lld is not a multiple of d1 = %lld", (long long)batch, (long long)d1);
  GemmParams p{};
  p.a = a;
  p.b = b;
  p.c = c;
  p.M = (int32_t)M;
  p.N = (int32_t)N;
  p.K = (int32_t)K;
  p.batch = (int32_t)batch;
  p.lda = lda;
  p.ldb = ldb;
  p.sa = stride_a;
  p.sb = stride_b;
  p.layout = layout;
  if (d1 > 0) {  // [B/d1, d1, M, N] -> [B/d1, M, d1, N]
    p.ldc = d1 * N;
    p.sc = N;
    p.batch_inner = (int32_t)d1;
    p.sc_outer = M * d1 * N;
  } else {
    p.ldc = ldc;
    p.sc = stride_c;
  }
  p.ldd = p.ldc;
  return run_gemm(kEpiNone, dtype, algo, p, reinterpret_cast<hipStream_t>(stream));
}

int aitamd_bmm_add(int layout, int dtype, int algo, const void* a, const void* b, const void* d0, void* c, int64_t batch,
                   int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t ldd,
                   int64_t stride_a, int64_t stride_b, int64_t stride_c, int64_t stride_d, void* stream) {
  if (layout < AITAMD_LAYOUT_RCR || layout > AITAMD_LAYOUT_CRR) return fail("aitamd_bmm_add: unknown layout %d", layout);
  if (M > 0x7fffffffll || N > 0x7fffffffll || K > 0x7fffffffll || batch > 0x7fffffffll)
    return fail("aitamd_bmm_add: dimension too large");
  if (M > 0 && N > 0 && batch > 0 && !d0) return fail("aitamd_bmm_add: the residual pointer is null");
  if (ldd < N) return fail("aitamd_bmm_add: residual pitch smaller than N");
  GemmParams p{};
  p.a = a;
  p.b = b;
  p.c = c;
  p.d0 = d0;
  p.M = (int32_t)M;
  p.N = (int32_t)N;
  p.K = (int32_t)K;
  p.batch = (int32_t)batch;
  p.lda = lda;
  p.ldb = ldb;
  p.ldc = ldc;
  p.ldd = ldd;
  p.sa = stride_a;
  p.sb = stride_b;
  p.sc = stride_c;
  p.sd = stride_d;
  p.layout = layout;
  return run_gemm(kEpiAdd, dtype, algo, p, reinterpret_cast<hipStream_t>(stream));
}

}  // extern "C"
