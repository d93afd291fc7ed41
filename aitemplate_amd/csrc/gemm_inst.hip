// One translation unit per (epilogue, dtype): compiled repeatedly by the
// Makefile with -DAITAMD_EPI=<EpilogueId> -DAITAMD_DT=<0 fp16 | 1 bf16>.
// It instantiates every tile of gemm_tiles.inc for that pair and exports the
// resulting launcher table under a C symbol the dispatcher looks up.
#include <cstdlib>
#include <mutex>
#include <type_traits>

#include "gemm_host.hpp"
#include "gemm_kernel_dma.hpp"
#include "gemm_kernel_persist.hpp"
#include "gemm_kernel_rows.hpp"
#include "gemm_kernel_wide.hpp"

#ifndef AITAMD_EPI
#error "compile with -DAITAMD_EPI=<id>"
#endif
#ifndef AITAMD_DT
#error "compile with -DAITAMD_DT=<0|1>"
#endif

namespace aitamd {
namespace {

#if AITAMD_DT == 0
using Elem = f16;
#define AITAMD_DT_NAME "f16"
#else
using Elem = bf16;
#define AITAMD_DT_NAME "bf16"
#endif

constexpr int kMaxDevices = 64;

using Epi = Epilogue<AITAMD_EPI>;

// Kernels with the permuted store exist for the two epilogues the permuting ops use.
constexpr bool kHasPermutedStore = AITAMD_EPI == kEpiNone || AITAMD_EPI == kEpiBias;

// Kernels for operands that are not K-contiguous exist on the direct-to-LDS tiles whose edges allow it, for the
// epilogues the reference's ops in those layouts use: plain and residual-add in all of rrr, ccr, crr; bias for
// rrr with the permuted store (gemm_rrr_bias_permute).  kLayoutBits: bit L set when layout L is compiled.
constexpr int kLayoutBits = (AITAMD_EPI == kEpiNone || AITAMD_EPI == kEpiAdd) ? 0xf : (AITAMD_EPI == kEpiBias ? 0x3 : 0x1);
constexpr bool kLayoutsArePermuted = AITAMD_EPI == kEpiBias;  // the bias kernels of the other layouts store permuted

constexpr int kShortK = 4;
template <class Tile, bool PERM, int LAYOUT>
struct KernelOf;
template <int BM, int BN, int BK, int WM, int WN, int NS, int OCC, int PIPE, int MT, int AUX, int MODE, bool PERM,
          int LAYOUT>
struct KernelOf<GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, AUX, MODE>, PERM, LAYOUT> {
  static constexpr auto value =
      gemm_rcr_dma_kernel<Elem, GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, AUX, MODE>, Epi, PERM, LAYOUT>;
};

template <int BM, int BN, int BK, int WM, int WN, int NS, int MT, int LBM, int PAIR, bool PERM, int LAYOUT>
struct KernelOf<GemmTilePersist<BM, BN, BK, WM, WN, NS, MT, LBM, PAIR>, PERM, LAYOUT> {
  // (LAYOUT 4 is not an operand layout: it names the instantiation for tiles of fewer K-slabs than ring stages)
  static constexpr auto value =
      gemm_rcr_persist_kernel<Elem, GemmTilePersist<BM, BN, BK, WM, WN, NS, MT, LBM, PAIR>, Epi, PERM, LAYOUT == kShortK>;
};
template <int NW, int NS, int ELEM, bool PERM, int LAYOUT>
struct KernelOf<GemmTileRows<NW, NS, ELEM>, PERM, LAYOUT> {
  static constexpr auto value = gemm_rcr_rows_kernel<Elem, GemmTileRows<NW, NS, ELEM>, Epi, PERM>;
};
template <int MI, int NI, int KTAIL, bool PERM, int LAYOUT>
struct KernelOf<GemmTileWide<MI, NI, KTAIL>, PERM, LAYOUT> {
  static constexpr auto value = gemm_rcr_wide_kernel<Elem, GemmTileWide<MI, NI, KTAIL>, Epi>;
};
// the slab-pair form of a persistent tile (the tile itself where it has none)
template <class Tile>
struct PairOf {
  using type = Tile;
};
template <int BM, int BN, int BK, int WM, int WN, int MT, int LBM>
struct PairOf<GemmTilePersist<BM, BN, BK, WM, WN, 4, MT, LBM, 0>> {
  using Plain = GemmTilePersist<BM, BN, BK, WM, WN, 4, MT, LBM, 0>;
  using type = std::conditional_t<Plain::kPairable,
                                  GemmTilePersist<BM, BN, BK, WM, WN, 5, MT, LBM, Plain::kPairable ? 1 : 0>, Plain>;
};
// bit L set: the tile has a kernel for layout L (bit 0, rcr, always)
template <class Tile>
struct LayoutMask {
  static constexpr int value = 1;
};
template <int BM, int BN, int BK, int WM, int WN, int NS, int OCC, int PIPE, int MT, int AUX>
struct LayoutMask<GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, AUX, 0>> {
  static constexpr int value =
      GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, AUX>::kTransposable ? kLayoutBits : 1;
};
// (the register-staged form takes every layout, pitch and K: the instances of last resort)
template <int BM, int BN, int BK, int WM, int WN, int NS, int OCC, int PIPE, int MT, int AUX>
struct LayoutMask<GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, AUX, 4>> {
  static constexpr int value =
      GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, AUX, 4>::kTransposable ? kLayoutBits : 1;
};
// split-K form: rcr only
template <class Tile>
struct IsSplitK {
  static constexpr bool value = false;
};
template <int BM, int BN, int BK, int WM, int WN, int NS, int OCC, int PIPE, int MT, int AUX, int MODE>
struct IsSplitK<GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, AUX, MODE>> {
  static constexpr bool value = (MODE & 1) != 0;
};
template <class Tile>
struct IsPersistent {
  static constexpr bool value = false;
};
template <int BM, int BN, int BK, int WM, int WN, int NS, int MT, int LBM, int PAIR>
struct IsPersistent<GemmTilePersist<BM, BN, BK, WM, WN, NS, MT, LBM, PAIR>> {
  static constexpr bool value = true;
};

template <class Tile>
struct IsWide {
  static constexpr bool value = false;
};
template <int MI, int NI, int KTAIL>
struct IsWide<GemmTileWide<MI, NI, KTAIL>> {
  static constexpr bool value = true;
};

template <class Tile>
struct IsRows {
  static constexpr bool value = false;
};
template <int NW, int NS, int ELEM>
struct IsRows<GemmTileRows<NW, NS, ELEM>> {
  static constexpr bool value = true;
};

// Workgroups per tile of a split-K launch (split_k_rule)
template <class Tile>
int split_k_factor(const GemmParams& p, int cus) {
  const int64_t tiles = (int64_t)((p.M + Tile::BM - 1) / Tile::BM) * ((p.N + Tile::BN - 1) / Tile::BN) * p.batch;
  const int64_t k_tiles = ((Tile::KVEC == 8 ? p.K : (p.K & ~7)) + Tile::BK - 1) / Tile::BK;
  return split_k_rule(tiles, k_tiles, Tile::BK, (int64_t)Tile::BM * Tile::BN, cus);
}
template <class Tile>
int64_t workspace_of(const GemmParams& p) {
  if constexpr (IsSplitK<Tile>::value) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    const int64_t tiles = (int64_t)((p.M + Tile::BM - 1) / Tile::BM) * ((p.N + Tile::BN - 1) / Tile::BN) * p.batch;
    const int s = split_k_factor<Tile>(p, device_cus(dev));
    return s > 1 ? Tile::ws_bytes(tiles, s) : 0;
  }
  return 0;
}

// The per-XCD block mapping of the persistent kernels (GemmParams::xcd_shift; -1: the grouped mapping).  The grid of
// one batch is cut into 2^xcd_shift column blocks times 8 / 2^xcd_shift row blocks, one per XCD,
// where it divides so and the B panels of a block's columns take at most 2.5 MiB; the fewest column blocks that fit
// are taken, which share an A panel among the most tiles.  An XCD then reads few B panels over and over and every
// A panel once.  Measured on M=24576 N=3072 K=768 (two column blocks of six tile columns): 158 MB fetched per launch
// against 176 MB with the grouped mapping, 0.5 % (normally distributed operands) to 2 % (constant ones) less time.
// The B panels do not stay in the 4 MiB L2 from one block row to the next all the same: a round of 32 tiles streams
// 4.4 MB of distinct panel data between two uses of a B line (loading A with the non-temporal policy to protect B
// loses the sharing of A among the tiles of a row: 0.159 against 0.123 ms).
inline int xcd_block_shift(const GemmParams& p, int64_t tiles_m, int64_t tiles_n, int bn, int64_t grid) {
  if (p.batch != 1 || grid % 8 != 0 || tiles_m <= 0 || tiles_n <= 0) return -1;
  for (int shift = 0; shift <= 3; ++shift) {
    if (tiles_n % (1 << shift) != 0 || tiles_m % (8 >> shift) != 0) continue;
    const int64_t b_bytes = (tiles_n >> shift) * bn * p.K * 2;
    if (b_bytes <= (5ll << 19)) return shift;
  }
  return -1;
}

template <class Tile, bool PERM, int LAYOUT = 0>
hipError_t launch_kernel(const GemmParams& p_in, hipStream_t stream) {
  auto kernel = KernelOf<Tile, PERM, LAYOUT>::value;
  // LDS above 64 KiB has to be opted into once per device.
  static std::once_flag once[kMaxDevices];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  // the outcome is kept per device: a failed opt-in must fail every later call too, not only the first
  static hipError_t attr_errs[kMaxDevices];
  hipError_t& attr_err = attr_errs[dev % kMaxDevices];
  std::call_once(once[dev % kMaxDevices], [&] {
    attr_err = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, Tile::kLdsBytes);
  });
  if (attr_err != hipSuccess) return attr_err;

  GemmParams p = p_in;
  // streaming stores for outputs that will not be cached anyway (the 8 L2s hold 32 MiB together); the
  // buffer form needs one batch of the output to span less than 2 GiB
  {
    static const long long nt_min = getenv("AITAMD_NT_MIN_BYTES") ? atoll(getenv("AITAMD_NT_MIN_BYTES")) : (32ll << 20);
    const long long span = p.perm_on ? (long long)p.M * p.N * 2 : ((long long)(p.M - 1) * p.ldc + p.N) * 2;
    p.nt_store = (long long)p.M * p.N * p.batch * 2 >= nt_min && span < 0x7fffffffll;
  }
  const int64_t tiles_m = ((int64_t)p.M + Tile::BM - 1) / Tile::BM, tiles_n = ((int64_t)p.N + Tile::BN - 1) / Tile::BN;
  if (tiles_m <= 0 || tiles_n <= 0 || p.batch <= 0) return hipSuccess;
  // one workgroup per (batch, tile) pair, or, for the persistent kernels, one per CU walking them
  if (tiles_m * tiles_n > 0x7fffffffll / p.batch) return hipErrorInvalidValue;
  const int64_t total = tiles_m * tiles_n * p.batch;
  dim3 grid((unsigned)total, 1, 1);
  if constexpr (IsPersistent<Tile>::value || IsWide<Tile>::value) {
    const int cus = device_cus(dev);
    grid = dim3((unsigned)(total < cus ? total : cus), 1, 1);
    // few tile columns: the grouped walk goes row by row, so that the run of tiles of an XCD ends inside at most
    // one row of tiles whose A panel a second XCD then fetches too (eight rows with the default group height;
    // measured on M=24576 N=768 K=3072 and M=12608 N=1024 K=4096: 1 % less time)
    // (the four-wave tiles: groups of four rows, so that more XCDs work on the same columns at a time; 8192^3 on the
    // metric's kind of operands 712 us against 731 with eight)
    set_tiles(p, Tile::BM, Tile::BN, tiles_n <= 4 ? 0 : (IsWide<Tile>::value ? 2 : 3),
              xcd_block_shift(p, tiles_m, tiles_n, Tile::BN, grid.x));
  } else {
    set_tiles(p, Tile::BM, Tile::BN, IsRows<Tile>::value ? 0 : 3, -1);
  }
  if constexpr (PERM) {
    p.by_perm_m1 = make_divisor(p.perm_m1);
    p.by_perm_m2 = make_divisor(p.perm_m2);
    p.by_perm_n1 = make_divisor(p.perm_n1);
    p.by_perm_n2 = make_divisor(p.perm_n2);
  }
  if constexpr (IsSplitK<Tile>::value) {
    // tiles are shared along K only with enough scratch memory to hold the partial tiles; without it the
    // instance runs as its plain counterpart (one workgroup per tile, nothing written to the scratch memory)
    p.split_k = split_k_factor<Tile>(p, device_cus(dev));
    if (p.ws == nullptr || p.ws_bytes < Tile::ws_bytes(total, p.split_k) || total * p.split_k > 0x7fffffffll)
      p.split_k = 1;
    grid = dim3((unsigned)(total * p.split_k), 1, 1);
  }
  hipLaunchKernelGGL(kernel, grid, dim3(Tile::NT), Tile::kLdsBytes, stream, p);
  return hipGetLastError();
}

template <class Tile>
hipError_t launch_tile(const GemmParams& p, hipStream_t stream) {
  if constexpr (IsWide<Tile>::value) {
    if (p.layout != 0) return hipErrorInvalidValue;
    const bool multiplies = four_waves_multiply(Tile::KVEC, p.K) && (p.N & 7) == 0;
    if (multiplies && four_waves_store(p)) return launch_kernel<Tile, false>(p, stream);
    // Asked for by name with others: an instance that takes the same operands, any K and any output.  For a permuted store
    // the one of the same matrix instructions, whose results are those of the plain store.
    if (multiplies && p.perm_on) return launch_tile<GemmTileDma<32, 32, 128, 2, 2, 4, 2, 0, 16, 0, Tile::KTAIL != 0 ? 2 : 0>>(p, stream);
    using Other = std::conditional_t<Tile::KTAIL != 0, GemmTileDma<128, 128, 64, 2, 4, 4, 1, 1, 32, 0, 2>,
                                     GemmTilePersist<256, 256, 32, 2, 4, 4, 16, 256>>;
    return launch_tile<Other>(p, stream);
  } else {
  if (p.layout != 0) {
    constexpr int mask = LayoutMask<Tile>::value;
    if ((p.perm_on != 0) != kLayoutsArePermuted) return hipErrorInvalidValue;
    if constexpr ((mask & 2) != 0) {
      if (p.layout == 1) return launch_kernel<Tile, kLayoutsArePermuted, 1>(p, stream);
    }
    if constexpr ((mask & 4) != 0) {
      if (p.layout == 2) return launch_kernel<Tile, kLayoutsArePermuted, 2>(p, stream);
    }
    if constexpr ((mask & 8) != 0) {
      if (p.layout == 3) return launch_kernel<Tile, kLayoutsArePermuted, 3>(p, stream);
    }
    return hipErrorInvalidValue;
  }
  if constexpr (IsPersistent<Tile>::value) {
    const int64_t k_tiles = ((int64_t)p.K + Tile::BK - 1) / Tile::BK;
    if (k_tiles < Tile::NS) {
      if (p.perm_on) {
        if constexpr (kHasPermutedStore) return launch_kernel<Tile, true, kShortK>(p, stream);
        return hipErrorInvalidValue;
      }
      return launch_kernel<Tile, false, kShortK>(p, stream);
    }
    // tiles of an even number of K-slabs go to the slab-pair form of the kernel where the tile has one: the same
    // products summed in the same order (the results are the same bit for bit), the loads better ordered
    using Pair = typename PairOf<Tile>::type;
    if constexpr (!std::is_same_v<Pair, Tile>) {
      // (AITAMD_NO_SLAB_PAIRS=1 keeps every tile on the one-slab form, for measuring one against the other)
      static const bool pairs_on = !(getenv("AITAMD_NO_SLAB_PAIRS") && atoi(getenv("AITAMD_NO_SLAB_PAIRS")) != 0);
      if (pairs_on && k_tiles % 2 == 0 && k_tiles >= Tile::kPairMinSlabs) {
        if (p.perm_on) {
          if constexpr (kHasPermutedStore) return launch_kernel<Pair, true>(p, stream);
          return hipErrorInvalidValue;
        }
        return launch_kernel<Pair, false>(p, stream);
      }
    }
  }
  if (p.perm_on) {
    if constexpr (kHasPermutedStore) return launch_kernel<Tile, true>(p, stream);
    return hipErrorInvalidValue;
  }
  return launch_kernel<Tile, false>(p, stream);
  }
}

// Workgroups one CU can hold: limited by LDS (160 KiB) and by the register file
// (512 VGPRs per SIMD lane shared by the waves of a SIMD).
constexpr int kLdsPerCu = 160 * 1024;
constexpr int dma_wgs_per_cu(int nt, int occ, int lds) {
  const int waves_per_wg_per_simd = nt / 64 / 4 > 0 ? nt / 64 / 4 : 1;
  const int by_regs = occ / waves_per_wg_per_simd > 0 ? occ / waves_per_wg_per_simd : 1;
  const int by_lds = kLdsPerCu / lds > 0 ? kLdsPerCu / lds : 1;
  return by_regs < by_lds ? by_regs : by_lds;
}

// Table entry of a tile.  KIND: GemmAlgo::direct_lds; OCC: workgroups per CU of the persistent and few-rows kernels,
// waves per SIMD that the registers allow of the others.
struct Cost {
  float start, mult, fetch, alone, tile;
};
template <class Tile, int KIND, int OCC>
constexpr GemmAlgo entry(const char* name, Cost c) {
  constexpr bool kByRegisters = KIND != 2 && KIND != 8 && KIND != 16;
  return {name, Tile::BM, Tile::BN, Tile::BK, Tile::NT, Tile::KVEC, Tile::kLdsBytes,
          kByRegisters ? dma_wgs_per_cu(Tile::NT, OCC, Tile::kLdsBytes) : OCC, KIND, LayoutMask<Tile>::value, &launch_tile<Tile>,
          KIND == 4 ? &workspace_of<Tile> : nullptr, {c.start, c.mult, c.fetch, c.alone, c.tile}};
}

const GemmAlgo kAlgos[] = {
#define AITAMD_NAME "gemm_rcr_" AITAMD_DT_NAME "_"
#define AITAMD_GEMM_TILE_DMA(BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, AUX, ...)                                        \
  entry<GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, AUX>, 1, OCC>(                                            \
      AITAMD_NAME #BM "x" #BN "x" #BK "_w" #WM "x" #WN "_dma" #NS "_o" #OCC "_p" #PIPE "_m" #MT "_c" #AUX, {__VA_ARGS__}),
#define AITAMD_GEMM_TILE_PERSIST(BM, BN, BK, WM, WN, NS, MT, LBM, ...)                                               \
  entry<GemmTilePersist<BM, BN, BK, WM, WN, NS, MT, LBM>, 2, 1>(                                                     \
      AITAMD_NAME #BM "x" #BN "x" #BK "_w" #WM "x" #WN "_persist" #NS "_m" #MT, {__VA_ARGS__}),
#define AITAMD_GEMM_TILE_WIDE(MI, NI, BM, BN, ...)                                                                   \
  entry<GemmTileWide<MI, NI, 0>, 16, 1>(AITAMD_NAME #BM "x" #BN "x32_w2x2_wide", {__VA_ARGS__}),
#define AITAMD_GEMM_TILE_WIDE_K2(MI, NI, BM, BN, ...)                                                                \
  entry<GemmTileWide<MI, NI, 1>, 16, 1>(AITAMD_NAME #BM "x" #BN "x32_w2x2_wide_k2", {__VA_ARGS__}),
#define AITAMD_GEMM_TILE_DMA_SPLITK(BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, ...)                                      \
  entry<GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, 0, 1>, 4, OCC>(                                           \
      AITAMD_NAME #BM "x" #BN "x" #BK "_w" #WM "x" #WN "_dma" #NS "_o" #OCC "_p" #PIPE "_m" #MT "_splitk", {__VA_ARGS__}),
#define AITAMD_GEMM_TILE_DMA_K2(BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, ...)                                          \
  entry<GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, 0, 2>, 1, OCC>(                                           \
      AITAMD_NAME #BM "x" #BN "x" #BK "_w" #WM "x" #WN "_dma" #NS "_o" #OCC "_p" #PIPE "_m" #MT "_k2", {__VA_ARGS__}),
#define AITAMD_GEMM_TILE_DMA_SPLITK_K2(BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, ...)                                   \
  entry<GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, PIPE, MT, 0, 3>, 4, OCC>(                                           \
      AITAMD_NAME #BM "x" #BN "x" #BK "_w" #WM "x" #WN "_dma" #NS "_o" #OCC "_p" #PIPE "_m" #MT "_k2_splitk", {__VA_ARGS__}),
#define AITAMD_GEMM_TILE_STAGED(BM, BN, BK, WM, WN, NS, OCC, MT, ...)                                                \
  entry<GemmTileDma<BM, BN, BK, WM, WN, NS, OCC, 0, MT, 0, 4>, 0, OCC>(                                              \
      AITAMD_NAME #BM "x" #BN "x" #BK "_w" #WM "x" #WN "_reg" #NS "_o" #OCC "_v1", {__VA_ARGS__}),
#define AITAMD_GEMM_ROWS(NW, NS, ...)                                                                                \
  entry<GemmTileRows<NW, NS, 0>, 8, 2>(AITAMD_NAME "rows16x16_n" #NW "_s" #NS "_k2", {__VA_ARGS__}),
#define AITAMD_GEMM_ROWS_ELEM(NW, NS, ...)                                                                           \
  entry<GemmTileRows<NW, NS, 1>, 8, 2>(AITAMD_NAME "rows16x16_n" #NW "_s" #NS "_v1", {__VA_ARGS__}),
#include "gemm_tiles.inc"
#undef AITAMD_GEMM_TILE_DMA
#undef AITAMD_GEMM_TILE_PERSIST
#undef AITAMD_GEMM_TILE_WIDE
#undef AITAMD_GEMM_TILE_WIDE_K2
#undef AITAMD_GEMM_TILE_DMA_SPLITK
#undef AITAMD_GEMM_TILE_DMA_K2
#undef AITAMD_GEMM_TILE_DMA_SPLITK_K2
#undef AITAMD_GEMM_TILE_STAGED
#undef AITAMD_GEMM_ROWS
#undef AITAMD_GEMM_ROWS_ELEM
#undef AITAMD_NAME
};

}  // namespace
}  // namespace aitamd

#define AITAMD_CAT3(a, b, c) a##b##_##c
#define AITAMD_TABLE_SYM(e, d) AITAMD_CAT3(aitamd_gemm_table_, e, d)

extern "C" __attribute__((visibility("hidden"))) aitamd::GemmAlgoTable AITAMD_TABLE_SYM(AITAMD_EPI, AITAMD_DT)() {
  return {aitamd::kAlgos, (int)(sizeof(aitamd::kAlgos) / sizeof(aitamd::kAlgos[0])), aitamd::Epi::kNumD};
}
