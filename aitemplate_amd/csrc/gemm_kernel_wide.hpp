// Persistent direct-to-LDS RCR GEMM on four waves: one wave per SIMD owns a quarter of a 256-row tile, its
// accumulators in the upper half of the 512 registers that a lane of it has.
//
// Against the eight-wave persistent kernel (gemm_kernel_persist.hpp), whose workgroup -> tile walk and slab-pair loads
// (16 rows of two K-slabs back to back, the halves of the same lines) it shares: a wave's part is 128 x 128 instead of
// 128 x 64, so a K-step reads 16 fragments for 64 MFMAs and not 12 for 32 - a third less LDS traffic, and energy, which
// is what large products run out of on this part.  A wave alone on its SIMD has nobody to hide behind, so
//  * the fragments of a K-step are read into a second set of registers during the step before, and a ring stage is
//    free for the slab five further on as soon as they have been;
//  * the loop is written instruction by instruction (volatile asm keeps the order): between two MFMAs, 16 cycles, there
//    is room for one other instruction, and each further one costs about 4.  The loop has 60 scalar and vector
//    instructions for 128 MFMAs; with the loads as builtins (an LDS base, a select and a wait state in front of each, the
//    ring arithmetic and two descriptors per pair) it had 180.  8192^3 on constant operands: 629 us with them, 567 now;
//    502 without the loads.  One branch per slot of the loop instead (to spread the four waves' loads): 879;
//  * MFMAs and their accumulators are asm with accumulation-register operands: left to itself the compiler copies
//    accumulators between the two halves of the register file inside the loop.
// What bounds it: the board's power on operands with random bits, the latency of lines from beyond the L2 on constant
// ones (where all come from the L2: 537 us).  A slab's loads over one K-step instead of two: 837 us against 715 (before
// the above); one slab at a time: 870; lines touched ahead of their loads, to bring them into the L2: no gain on random
// operands.  8192^3 bf16, normally distributed operands: 813 us (eight waves) -> 721.
//
// The epilogue needs no LDS: v_permlane16_swap between two column blocks gives a lane 8 consecutive columns of a row,
// in fp32.  It stores 16-byte pieces through buffer descriptors only; the launcher sends other outputs elsewhere.
#pragma once

#include <type_traits>

#include "gemm_kernel_dma.hpp"

namespace aitamd {

// KTAIL_: K, row pitches and operand pointers in whole dwords (MODE bit 1 of GemmTileDma): the slabs cover K's whole
// 16-byte pieces and the up to three dwords behind them are loaded straight into MFMA operands after the loop.
template <int MI_, int NI_, int KTAIL_ = 0>
struct GemmTileWide {
  static constexpr int MI = MI_, NI = NI_, KTAIL = KTAIL_;  // 16 x 16 blocks of a wave's part
  static constexpr int WTM = 16 * MI, WTN = 16 * NI;
  static constexpr int BM = 2 * WTM, BN = 2 * WTN;
  static constexpr int BK = 32;                    // K of one slab, one step of the 16x16x32 MFMA
  static constexpr int KVEC = KTAIL ? 2 : 8;
  static constexpr int NS = 5;                     // ring stages
  static constexpr int NW = 4, NT = NW * kWaveSize;
  static constexpr int RA = 256, RB = 256;         // rows of A and of B that a stage holds
  static constexpr int STAGE_BYTES = (RA + RB) * BK * 2;
  static constexpr int kLdsBytes = NS * STAGE_BYTES;
  static_assert(BM <= RA && BN <= RB && MI % 2 == 0, "the tile's rows fit a stage");
  static_assert(kLdsBytes <= 160 * 1024, "LDS budget");
};

// Matrix instructions on accumulators in the accumulation registers
template <class T>
struct AccMfma;
template <>
struct AccMfma<f16> {
  static AITAMD_DEVICE void run(f32x4& c, f16x8 a, f16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  static AITAMD_DEVICE void first(f32x4& c, f16x8 a, f16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  }
};
template <>
struct AccMfma<bf16> {
  static AITAMD_DEVICE void run(f32x4& c, bf16x8 a, bf16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  static AITAMD_DEVICE void first(f32x4& c, bf16x8 a, bf16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  }
};

template <int OFF, class V>
AITAMD_DEVICE void lds_read16(V& v, uint32_t addr) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
}

// odd 16-lane rows of x exchanged with the even ones of y
AITAMD_DEVICE void swap_rows16(float& x, float& y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  x = __uint_as_float(r[0]);
  y = __uint_as_float(r[1]);
}

// x of lanes 8 .. 15 of every 16 exchanged with y of lanes 0 .. 7
AITAMD_DEVICE void swap_halves16(uint32_t& x, uint32_t& y) {
  constexpr int kRowRor8 = 0x128;
  const uint32_t nx = __builtin_amdgcn_update_dpp(x, y, kRowRor8, 0xf, 0xc, false);
  y = __builtin_amdgcn_update_dpp(y, x, kRowRor8, 0xf, 0x3, false);
  x = nx;
}

template <class T, class Tile, class Epi>
__global__ void __launch_bounds__(Tile::NT, 1) gemm_rcr_wide_kernel(const GemmParams p) {
  using Tr = ElemTraits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int BM = Tile::BM, BN = Tile::BN, NS = Tile::NS, MI = Tile::MI, NI = Tile::NI;
  constexpr int STAGE = Tile::STAGE_BYTES;
  constexpr int SLAB = Tile::BK * 2;  // bytes of a row in one slab
  typedef __attribute__((address_space(3))) void lds_void;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 15, fq = lane >> 4;

  const int total_tiles = p.tiles_m * p.tiles_n * p.batch;
  const int G = gridDim.x, g = blockIdx.x;
  const int k_main = Tile::KTAIL ? (p.K & ~7) : p.K;
  // slab pairs of a tile (K > 128: the loop is built of three at least), and the bytes of K in the last one
  const int n_pairs = (k_main + 2 * Tile::BK - 1) / (2 * Tile::BK);
  const int tail_bytes = k_main * 2 - (n_pairs - 1) * 2 * SLAB;
  const int my_tiles = (total_tiles - g + G - 1) / G;

  struct TileCoord {
    int m0, n0, batch;
  };
  auto tile_coord = [&](int i) __attribute__((always_inline)) {
    TileCoord c;
    int b, tm, tn;
    map_tile<true>(p, g + i * G, b, tm, tn);
    c.m0 = tm * BM;
    c.n0 = tn * BN;
    c.batch = b;
    return c;
  };

  // ---- loader ----
  const bool loads_a = wave < 2;
  const int l_row = lane >> 2;
  const int l_chunk = (lane & 3) ^ ((lane >> 3) & 3);
  const int64_t l_ld = loads_a ? p.lda : p.ldb;
  // Byte offsets of the lane's 16 bytes of the wave's eight blocks (16 rows each) in slabs a and b of a pair.  Two blocks
  // share an LDS base: the second is placed by the load's immediate offset, which its lane offset takes back.
  uint32_t off_a[8], off_b[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    off_a[i] = (uint32_t)((((wave & 1) * 128 + i * 16 + l_row) * l_ld) * 2 + l_chunk * 16 - (i & 1) * 1024);
    off_b[i] = off_a[i] + SLAB;
  }

  struct Panel {
    uint32_t lo, hi, bytes;
  };
  auto tile_panel = [&](int i) __attribute__((always_inline)) {
    Panel q;
    const void* base = p.a;
    uint32_t bytes = 0;
    if (i < my_tiles) {
      const TileCoord c = tile_coord(i);
      const int rows_a = (p.M - c.m0) < BM ? (p.M - c.m0) : BM;
      const int rows_b = (p.N - c.n0) < BN ? (p.N - c.n0) : BN;
      const T* Ab = reinterpret_cast<const T*>(p.a) + (int64_t)c.batch * p.sa + (int64_t)c.m0 * p.lda;
      const T* Bb = reinterpret_cast<const T*>(p.b) + (int64_t)c.batch * p.sb + (int64_t)c.n0 * p.ldb;
      const uint32_t bytes_a = clamp_records((((int64_t)rows_a - 1) * p.lda + p.K) * 2);
      const uint32_t bytes_b = clamp_records((((int64_t)rows_b - 1) * p.ldb + p.K) * 2);
      base = loads_a ? (const void*)Ab : (const void*)Bb;
      bytes = loads_a ? bytes_a : bytes_b;
    }
    const uint64_t v = reinterpret_cast<uint64_t>(base);
    q.lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    q.hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    q.bytes = __builtin_amdgcn_readfirstlane(bytes);
    return q;
  };
  // the panel's buffer from byte kb of its rows on
  auto panel_rsrc = [&](const Panel& q, int kb) __attribute__((always_inline)) {
    const uint64_t a = (((uint64_t)q.hi << 32) | q.lo) + (uint32_t)kb;
    const int left = (int)q.bytes - kb;
    return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, (uint32_t)(left > 0 ? left : 0), 0x00020000u};
  };
  // K ends inside a pair: its loads are out of range for the lanes past the end, by the top bit of their offsets
  const uint32_t past_a = l_chunk * 16 < tail_bytes ? 0u : kOobOffset;
  const uint32_t past_b = l_chunk * 16 + SLAB < tail_bytes ? 0u : kOobOffset;
  auto toggle_tail = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      off_a[i] ^= past_a;
      off_b[i] ^= past_b;
    }
  };
  auto set_m0 = [&](uint32_t base, auto i_c) __attribute__((always_inline)) {
    asm volatile("s_add_u32 m0, %0, %1" ::"s"(base), "n"(decltype(i_c)::value * 1024) : "memory", "scc");
  };
  auto load_lds = [&](uint32_t off, const u32x4& d, auto second_c) __attribute__((always_inline)) {
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen offset:%2 lds" ::"v"(off), "s"(d), "n"(decltype(second_c)::value * 1024) : "memory");
  };
  // ---- fragments ----
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void*)smem_raw;
  const uint32_t rd_lane = (uint32_t)(fr * 64 + ((fq ^ ((fr >> 1) & 3)) << 4));
  const uint32_t a_rd = lds0 + rd_lane + wm * Tile::WTM * 64;
  const uint32_t b_rd = lds0 + rd_lane + Tile::RA * 64 + wn * Tile::WTN * 64;
  f32x4 acc[MI][NI];
  vec8 fa0[MI], fb0[NI], fa1[MI], fb1[NI];

  // One K-step: the MFMAs on (a, b), between them the reads of the next step's fragments (one behind every second MFMA,
  // from ring stage `next`) and whatever else between() puts there.
  constexpr int READS = MI + NI;
  auto step = [&](auto first_c, vec8* a, vec8* b, vec8* na, vec8* nb, uint32_t next, auto&& between) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_c)::value;
    const uint32_t ra = a_rd + next, rb = b_rd + next;
    static_for<0, MI * NI>([&](auto x_c) __attribute__((always_inline)) {
      constexpr int x = decltype(x_c)::value;
      constexpr int ni = x / MI, mi = x % MI;
      if constexpr (FIRST)
        AccMfma<T>::first(acc[mi][ni], b[ni], a[mi]);
      else
        AccMfma<T>::run(acc[mi][ni], b[ni], a[mi]);
      if constexpr (x % 2 == 0 && x / 2 < READS) {
        constexpr int r = x / 2;
        if constexpr (r < NI)
          lds_read16<r * 1024>(nb[r], rb);
        else
          lds_read16<(r - NI) * 1024>(na[r - NI], ra);
      }
      between(x_c);
    });
  };
  // A slab pair (a, b), a even, slab t in ring stage t % 5.  Step a: behind its barrier every wave has read its fragments
  // of a (and of the slab before), so those two stages take the slabs a + 4 and a + 5, four of the wave's blocks in each
  // step.  Step b: behind its barrier the slabs a + 2 and a + 3 have landed - of the wave's loads only the eight of
  // step a are younger - and every wave has read its fragments of b.
  // ring stages as byte offsets: of the pair's first slab, of the slab before it, and of the two behind it
  uint32_t s0 = 0, sp = 4 * STAGE, s1 = STAGE, s2 = 2 * STAGE;
  const uint32_t m_wave = lds0 + wave * 8192;
  auto pair = [&](auto first_c, const u32x4& d) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_c)::value;
    const uint32_t ma = m_wave + sp, mb = m_wave + s0;
    // The loads' instructions between the MFMAs of a step: blocks B0 .. B0 + 3, a's and b's back to back.  The LDS base
    // is written two MFMAs ahead of the load.
    auto ld = [&](auto b0_c, auto x_c) __attribute__((always_inline)) {
      constexpr int PER = MI * NI / 4;
      constexpr int x = decltype(x_c)::value % PER;
      constexpr int i = decltype(b0_c)::value + decltype(x_c)::value / PER;
      constexpr std::integral_constant<int, (i & ~1)> base{};
      constexpr std::integral_constant<int, i % 2> second{};
      if constexpr (x == 5) set_m0(ma, base);
      if constexpr (x == 7) load_lds(off_a[i], d, second);
      if constexpr (x == 9) set_m0(mb, base);
      if constexpr (x == 11) load_lds(off_b[i], d, second);
    };
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    step(first_c, fa0, fb0, fa1, fb1, s1, [&](auto x_c) __attribute__((always_inline)) { ld(std::integral_constant<int, 0>{}, x_c); });
    if constexpr (FIRST)  // (landed before the stores of the tile before, which would be waited for as well)
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    step(std::false_type{}, fa1, fb1, fa0, fb0, s2, [&](auto x_c) __attribute__((always_inline)) { ld(std::integral_constant<int, 4>{}, x_c); });
    sp = s1;
    s0 = s2;
    s1 = s0 == 4 * STAGE ? 0 : s0 + STAGE;
    s2 = s1 == 4 * STAGE ? 0 : s1 + STAGE;
  };

  // ---- epilogue ----
  const T* bias = reinterpret_cast<const T*>(p.bias);
  // A lane's place in a pair of column blocks and in a pair of row blocks (the last column block of an odd number)
  const int sub = fq & 1, half8 = (fq >> 1) * 8;
  constexpr int NP = NI / 2;
  constexpr int NU = NP + (NI & 1);  // units (8 columns of a lane) per row block, or per two for the last one

  // f(x, y, row, unit): the accumulators whose exchange gives the lane 8 columns of a row
  auto for_units = [&](auto mp_c, auto&& f) __attribute__((always_inline)) {
    constexpr int mp = decltype(mp_c)::value;
    static_for<0, 2>([&](auto h_c) __attribute__((always_inline)) {
      constexpr int mi = 2 * mp + decltype(h_c)::value;
      static_for<0, NP>([&](auto u_c) __attribute__((always_inline)) {
        constexpr int u = decltype(u_c)::value;
        f(acc[mi][2 * u], acc[mi][2 * u + 1], std::integral_constant<int, (mi * NU + u) % (2 * NU)>{}, mi * 16, u_c);
      });
    });
    if constexpr (NI & 1) f(acc[2 * mp][NI - 1], acc[2 * mp + 1][NI - 1], std::integral_constant<int, 2 * NU - 1>{}, 2 * mp * 16, std::integral_constant<int, NP>{});
  };

  auto epilogue_as = [&](const TileCoord& c, auto nt_bits) __attribute__((always_inline)) {
    constexpr int NT_BITS = decltype(nt_bits)::value;
    const int m_w = c.m0 + wm * Tile::WTM;
    const int n_w = c.n0 + wn * Tile::WTN;
    const int rows_left = p.M - m_w;
    const uint32_t rows_valid = rows_left <= 0 ? 0u : (uint32_t)(rows_left < Tile::WTM ? rows_left : Tile::WTM);
    T* Cw = reinterpret_cast<T*>(p.c) + out_batch_offset(p, c.batch) + (int64_t)m_w * p.ldc + n_w;
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(Cw, rows_valid * (uint32_t)p.ldc * 2u);
    __amdgpu_buffer_rsrc_t rd0 = rc, rd1 = rc;
    if constexpr (Epi::kNumD >= 1)
      rd0 = make_rsrc(reinterpret_cast<const T*>(p.d0) + (int64_t)c.batch * p.sd + (int64_t)m_w * p.ldd + n_w, rows_valid * (uint32_t)p.ldd * 2u);
    if constexpr (Epi::kNumD >= 2)
      rd1 = make_rsrc(reinterpret_cast<const T*>(p.d1) + (int64_t)c.batch * p.sd + (int64_t)m_w * p.ldd + n_w, rows_valid * (uint32_t)p.ldd * 2u);
    // byte offsets of the lane's first row in each unit, out of range where its columns are; of a pair of units the
    // lane's share behind the exchange (below)
    uint32_t off_c[NU], off_d[NU];
    vec8 bv[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const bool row_pair = u == NP;
      const int col = u * 32 + (row_pair ? 0 : sub * 16) + half8;
      const int row = fr + (row_pair ? sub * 16 : 0);
      const bool ok = n_w + col < p.N;
      off_d[u] = ok ? (uint32_t)((row * (int)p.ldd + col) * 2) : kOobOffset;
      const bool joined = u < NP / 2 * 2;
      const int col_c = joined ? (u / 2 * 2 + (fr >> 3)) * 32 + sub * 16 + half8 : col;
      const int row_c = joined ? (fr & 7) + (u & 1) * 8 : row;
      off_c[u] = n_w + col_c < p.N ? (uint32_t)((row_c * (int)p.ldc + col_c) * 2) : kOobOffset;
      bv[u] = vec8{};
      if constexpr (Epi::kHasBias) {
        if (ok) bv[u] = load_vec<vec8>(bias + n_w + col);
      }
    }
    float one = 1.0f;
    asm volatile("" : "+s"(one));
    // (one residual: a row pair ahead of its use, and ahead of the stores of the pair before - loads and stores complete
    // in order, a load behind them waits for them; two of them held so spill)
    constexpr int AHEAD = Epi::kNumD == 1 ? 1 : 0;
    vec8 d0r[1 + AHEAD][2 * NU], d1r[1 + AHEAD][2 * NU];
    auto load_d = [&](auto mp_c) __attribute__((always_inline)) {
      constexpr int mp = decltype(mp_c)::value;
      if constexpr (Epi::kNumD >= 1 && mp < MI / 2) {
        for_units(mp_c, [&](const f32x4&, const f32x4&, auto s_c, int row, auto u_c) __attribute__((always_inline)) {
          const uint32_t off = off_d[decltype(u_c)::value] + (uint32_t)(row * (int)p.ldd * 2);
          d0r[mp % (1 + AHEAD)][decltype(s_c)::value] = __builtin_bit_cast(vec8, buffer_load_16B(rd0, off));
          if constexpr (Epi::kNumD >= 2) d1r[mp % (1 + AHEAD)][decltype(s_c)::value] = __builtin_bit_cast(vec8, buffer_load_16B(rd1, off));
        });
      }
    };
    if constexpr (AHEAD > 0) load_d(std::integral_constant<int, 0>{});
    static_for<0, MI / 2>([&](auto mp_c) __attribute__((always_inline)) {
      load_d(std::integral_constant<int, decltype(mp_c)::value + AHEAD>{});
      u32x4 held = {};
      const vec8 *d0v = d0r[decltype(mp_c)::value % (1 + AHEAD)], *d1v = d1r[decltype(mp_c)::value % (1 + AHEAD)];
      for_units(mp_c, [&](const f32x4& x, const f32x4& y, auto s_c, int row, auto u_c) __attribute__((always_inline)) {
        constexpr int u = decltype(u_c)::value, s = decltype(s_c)::value;
        float v[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = x[j];
          v[4 + j] = y[j];
          swap_rows16(v[j], v[4 + j]);
        }
        const vec8 o = epilogue8<Epi, T>(v, bv[u], d0v[s], d1v[s], one);
        auto store = [&](u32x4 v, uint32_t off) __attribute__((always_inline)) {
          __builtin_amdgcn_raw_buffer_store_b128(v, rc, off + (uint32_t)(row * (int)p.ldc * 2), 0, NT_BITS);
        };
        u32x4 w = __builtin_bit_cast(u32x4, o);
        // Two units are 128 bytes of 16 rows, 64 of each in a lane's four neighbours: exchanged so that eight lanes hold
        // the 128 bytes of a row: streaming stores of half a line each cost 2 us a round more (24576 x 2048, K = 768)
        if constexpr (u < NP / 2 * 2 && u % 2 == 0) {
          held = w;
        } else if constexpr (u < NP / 2 * 2) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            uint32_t lo = held[j], hi = w[j];
            swap_halves16(lo, hi);
            held[j] = lo;
            w[j] = hi;
          }
          store(held, off_c[u - 1]);
          store(w, off_c[u]);
        } else {
          store(w, off_c[u]);
        }
      });
    });
  };

  auto epilogue = [&](const TileCoord& c) __attribute__((always_inline)) {
    if (p.nt_store)
      epilogue_as(c, std::integral_constant<int, 2>{});
    else
      epilogue_as(c, std::integral_constant<int, 0>{});
  };

  // ---- tiles ----
  Panel nxt_p = tile_panel(0);
  const bool tail = tail_bytes < 2 * SLAB;
#pragma unroll
  for (int pr = 0; pr < 2; ++pr) {
    const u32x4 d = panel_rsrc(nxt_p, pr * 2 * SLAB);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" ::"s"(m_wave + pr * 2 * STAGE + (i & ~1) * 1024) : "memory");
      if (i & 1)
        load_lds(off_a[i], d, std::integral_constant<int, 1>{});
      else
        load_lds(off_a[i], d, std::integral_constant<int, 0>{});
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" ::"s"(m_wave + (pr * 2 + 1) * STAGE + (i & ~1) * 1024) : "memory");
      if (i & 1)
        load_lds(off_b[i], d, std::integral_constant<int, 1>{});
      else
        load_lds(off_b[i], d, std::integral_constant<int, 0>{});
    }
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  static_for<0, NI>([&](auto r_c) { lds_read16<decltype(r_c)::value * 1024>(fb0[decltype(r_c)::value], b_rd); });
  static_for<0, MI>([&](auto r_c) { lds_read16<decltype(r_c)::value * 1024>(fa0[decltype(r_c)::value], a_rd); });
  for (int i = 0; i < my_tiles; ++i) {
    const TileCoord cur = tile_coord(i);
    u32x4 d = panel_rsrc(nxt_p, 4 * SLAB);
    nxt_p = tile_panel(i + 1);
    // pair j is multiplied while pair j + 2 is requested: the tile's own up to its last, then the next tile's first two
    if (tail && n_pairs == 3) toggle_tail();
    pair(std::true_type{}, d);
    for (int j = 1; j < n_pairs - 2; ++j) {
      const uint64_t base = (((uint64_t)d[1] << 32) | d[0]) + 2 * SLAB;
      d[0] = (uint32_t)base;
      d[1] = (uint32_t)(base >> 32);
      d[2] -= 2 * SLAB;
      if (tail && j == n_pairs - 3) toggle_tail();
      pair(std::false_type{}, d);
    }
    if (tail) toggle_tail();
    for (int h = 0; h < 2; ++h) pair(std::false_type{}, panel_rsrc(nxt_p, h * 2 * SLAB));
    // (the results of the last matrix instructions are read no earlier than this; the next tile's first slabs, requested
    // before the stores that follow, have landed)
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    if constexpr (Tile::KTAIL != 0) {
      if (k_main < p.K) {
        // the up to three dwords behind the last whole 16-byte piece of each operand row
        const T* Ab = reinterpret_cast<const T*>(p.a) + (int64_t)cur.batch * p.sa + (int64_t)cur.m0 * p.lda;
        const T* Bb = reinterpret_cast<const T*>(p.b) + (int64_t)cur.batch * p.sb + (int64_t)cur.n0 * p.ldb;
        const int rows_a = (p.M - cur.m0) < BM ? (p.M - cur.m0) : BM;
        const int rows_b = (p.N - cur.n0) < BN ? (p.N - cur.n0) : BN;
        const __amdgpu_buffer_rsrc_t ra = make_rsrc(Ab, clamp_records((((int64_t)rows_a - 1) * p.lda + p.K) * 2));
        const __amdgpu_buffer_rsrc_t rb = make_rsrc(Bb, clamp_records((((int64_t)rows_b - 1) * p.ldb + p.K) * 2));
        // (opaque: offsets computed once for all tiles would be spilled, while the first tile's fragments are on their way)
        auto tail = [&](auto n_c, vec8* t, const __amdgpu_buffer_rsrc_t& r, int row, int64_t ld) __attribute__((always_inline)) {
          uint32_t at = (uint32_t)((row * (int)ld + k_main) * 2), zero = 0;
          asm volatile("" : "+v"(at), "+v"(zero));
          uint32_t off[3];
#pragma unroll
          for (int d = 0; d < 3; ++d) off[d] = fq == 0 && k_main + 2 * d < p.K ? at + 4 * d : kOobOffset;
#pragma unroll
          for (int i = 0; i < decltype(n_c)::value; ++i) {
            const uint32_t rows = (uint32_t)(i * 16 * (int)ld * 2);
            t[i] = __builtin_bit_cast(vec8, u32x4{buffer_load_4B(r, off[0] + rows), buffer_load_4B(r, off[1] + rows), buffer_load_4B(r, off[2] + rows), zero});
          }
        };
        vec8 ta[MI], tb[NI];
        tail(std::integral_constant<int, MI>{}, ta, ra, wm * Tile::WTM + fr, p.lda);
        tail(std::integral_constant<int, NI>{}, tb, rb, wn * Tile::WTN + fr, p.ldb);
        asm volatile("s_nop 7" ::: "memory");
        static_for<0, MI * NI>([&](auto x_c) __attribute__((always_inline)) {
          constexpr int x = decltype(x_c)::value;
          AccMfma<T>::run(acc[x % MI][x / MI], tb[x / MI], ta[x % MI]);
        });
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
      }
    }
    epilogue(cur);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

}  // namespace aitamd
