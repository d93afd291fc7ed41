// RCR GEMM for products of few output elements: 16 x 16 of them per workgroup, every wave on its own part of K.
//
// Bound: HBM for weights of many columns, one CU's share of the operand bytes for weights of few (a CU fetches about
// 45 bytes per clock), a trip to memory for the smallest.  The NW waves of a workgroup share K: wave w takes the 128-deep
// groups w, w + NW, ..., and fetches each straight to a ring in LDS that is its own: there is no barrier in the loop, and a
// wave waits for nothing but its oldest group.  v_mfma_f32_16x16x32 takes the 16 weight rows as one operand and 16 rows of
// A as the other; the waves' partial tiles are added through LDS in wave order.
//
// Through LDS and not to registers, where an operand's layout has 16 neighbouring lanes in 16 rows: a cache line per lane
// and 60 to 80 clocks per load, whatever the rows' alignment and however many are on their way.  To LDS 16 lanes fetch 256
// bytes of a row.  us, the register form with eight waves / this one:
//   1 x 768 x 768 3.9 / 3.4     2 x 432 x 6592 10.5 / 6.4     9 x 112 x 4736 10.2 / 5.8     4 x 288 x 4640 8.1 / 5.4
//   16 x 128 x 6480 13.4 / 8.2  1 x 6912 x 8314 23.2 / 22.7 (5.0 TB/s, as a large copy)  1 x 6912 x 8313 26.7 / 25.0
//   4 x 89 x 7425 13.2 / 7.5    14 x 201 x 8223 14.0 / 9.6
// and, against the tiles that took them, 16 x 2304 x 1024 5.3 / 4.1, 32 x 512 x 2048 6.9 / 4.5, 64 x 1024 x 1024 5.4 / 4.1,
// 31 x 1232 x 5504 14.0 / 9.5, 41 x 158 x 3879 9.3 / 6.8.  Tiles of 16 x 32, 32 x 16 and 32 x 32: slower at all of these.
// Groups past a wave's last are not requested - though out of range, their loads and the wait for them took 0.2 us of every launch -
// and the loop over all groups but the last ones has nothing to cut.  Before / after, on average over 40 to 70 problems each:
// M 5 to 16, K 65 to 128 2.97 / 2.70, K 513 to 1024 3.38 / 3.02, K above 4096 6.42 / 5.89; M to 4 at an odd K of 65 to 128 3.01 / 2.95,
// where the register form, without a pass through LDS, took 2.72.
// Four waves with two groups each on their way, or eight with one: two workgroups fit a CU (one, with twice as much on its
// way: as fast or up to a quarter slower).  Eight for odd elements, whose shifts a lone wave on its SIMD waits for.
//
// Any K, pitch and alignment (ELEM; else dwords).  Rows at odd elements are fetched from the dword they start in and put
// together by shifts of a piece and the dword behind it; that dword is in the next piece, so the last of a group's 16
// pieces serves the one before it only, and a group is 120 deep.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "epilogue.hpp"
#include "gemm_kernel.hpp"

namespace aitamd {

// NW_: waves; NS_: groups of a wave on their way; ELEM_: rows at any element, 0: at dwords
template <int NW_, int NS_, int ELEM_>
struct GemmTileRows {
  static constexpr int NW = NW_, NS = NS_, ELEM = ELEM_;
  static constexpr int BM = 16, BN = 16;
  static constexpr int GROUP = ELEM ? 120 : 128;  // K of a group
  static constexpr int BK = GROUP * NW;           // (what the waves take together)
  static constexpr int NT = NW * kWaveSize;
  static constexpr int KVEC = ELEM ? 1 : 2;
  static constexpr int STAGE = (BM + BN) * 256;  // bytes
  static constexpr int kRing = NW * NS * STAGE;
  static constexpr int kLdsBytes = kRing + (ELEM ? 16 : 0);  // (sixteen zeros)
  static_assert(NW * BM * BN * 4 <= kRing, "the partial tiles take the ring's place");
};

AITAMD_DEVICE void rows_load_lds(uint32_t lds, uint32_t off, const u32x4& desc) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(off), "s"(desc) : "memory");
}
AITAMD_DEVICE void rows_read16(u32x4& v, uint32_t at) { asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(at) : "memory"); }
AITAMD_DEVICE void rows_read4(uint32_t& v, uint32_t at) { asm volatile("ds_read_b32 %0, %1" : "=v"(v) : "v"(at) : "memory"); }
// what is read is there only behind the wait
AITAMD_DEVICE void rows_arrived(u32x4& v, uint32_t& behind) { asm volatile("" : "+v"(v), "+v"(behind)); }

template <class T, class Tile, class Epi, bool PERM = false>
__global__ void __launch_bounds__(Tile::NT) gemm_rcr_rows_kernel(const GemmParams p) {
  using Tr = ElemTraits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int NW = Tile::NW, NS = Tile::NS, BM = Tile::BM, BN = Tile::BN, GROUP = Tile::GROUP, ELEM = Tile::ELEM;
  typedef __attribute__((address_space(3))) void lds_void;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fq = lane >> 4;
  fetch_arguments(p);
  // tiles in rows: by_group divides by tiles_n
  const int batch = p.batch > 1 ? quotient((int)blockIdx.x, p.by_batch) : 0;
  const int id = (int)blockIdx.x - batch * (p.tiles_m * p.tiles_n);
  const int tm = quotient(id, p.by_group);
  const int m0 = tm * BM, n0 = (id - tm * p.tiles_n) * BN;
  const int rows_a = (p.M - m0) < BM ? (p.M - m0) : BM;
  const int rows_b = (p.N - n0) < BN ? (p.N - n0) : BN;

  const T* Ab = reinterpret_cast<const T*>(p.a) + (int64_t)batch * p.sa + (int64_t)m0 * p.lda;
  const T* Bb = reinterpret_cast<const T*>(p.b) + (int64_t)batch * p.sb + (int64_t)n0 * p.ldb;
  // (from the dword that the first row starts in to the one that the last row ends in)
  const uint32_t odd[2] = {(uint32_t)(reinterpret_cast<uintptr_t>(Ab) & 3), (uint32_t)(reinterpret_cast<uintptr_t>(Bb) & 3)};
  auto rsrc = [&](const T* base, uint32_t start, int rows, int64_t ld) __attribute__((always_inline)) {
    const uint64_t a = reinterpret_cast<uint64_t>(base) - start;
    const uint32_t bytes = clamp_records(((((int64_t)rows - 1) * ld + p.K) * 2 + start + 3) & ~3ll);
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu),
                 (uint32_t)__builtin_amdgcn_readfirstlane(bytes), 0x00020000u};
  };
  const u32x4 desc[2] = {rsrc(Ab, odd[0], rows_a, p.lda), rsrc(Bb, odd[1], rows_b, p.ldb)};

  // ---- loader: a load is 256 bytes, 16 pieces, of four rows.  Row r's piece c lies at place c ^ r of the row's 256 bytes
  // in LDS, so that the 16 rows of a fragment read are on different banks.
  const uint32_t pitch[2] = {(uint32_t)p.lda * 2u, (uint32_t)p.ldb * 2u};  // (a tile's rows span less than 2 GiB)
  uint32_t off[2][4], shift[2];
  int piece[4];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const uint32_t at0 = (uint32_t)(lane >> 4) * pitch[x] + odd[x];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      piece[i] = (lane & 15) ^ (i * 4 + (lane >> 4));
      const uint32_t at = at0 + (uint32_t)i * 4u * pitch[x];
      off[x][i] = (ELEM ? at & ~3u : at) + (uint32_t)piece[i] * 16u;
    }
    // (of row fr: the bits that its first element is behind the dword it lies in)
    shift[x] = (((uint32_t)fr * pitch[x] + odd[x]) & 2u) * 8u;
  }
  const uint32_t ring = (uint32_t)(uintptr_t)(lds_void*)smem_raw + wave * (NS * Tile::STAGE);
  const uint32_t zeros = (uint32_t)(uintptr_t)(lds_void*)smem_raw + Tile::kRing;
  if constexpr (ELEM != 0) {
    // (every wave writes them: it waits for nothing but its own)
    if (lane < 4) *reinterpret_cast<volatile uint32_t*>(smem_raw + Tile::kRing + lane * 4) = 0u;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  const int groups = (p.K + GROUP - 1) / GROUP;
  const int mine = (groups - wave + NW - 1) / NW;

  // a thread's outputs, and what the epilogue reads for them
  const int out_m = tid / BN, out_n = tid % BN;
  constexpr int OUTS = (BM * BN + Tile::NT - 1) / Tile::NT;
  T bias_v[OUTS], d0_v[OUTS], d1_v[OUTS];
  // (for an output that does not exist, of one that does: a branch around the loads would wait for them)
  auto read_epilogue = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int o = 0; o < OUTS; ++o) {
      const int m = out_m + o * (Tile::NT / BN);
      const int mc = m0 + (m < rows_a ? m : rows_a - 1), nc = n0 + (out_n < rows_b ? out_n : rows_b - 1);
      const int64_t at = (int64_t)batch * p.sd + (int64_t)mc * p.ldd + nc;
      bias_v[o] = d0_v[o] = d1_v[o] = T{};
      if constexpr (Epi::kHasBias) bias_v[o] = reinterpret_cast<const T*>(p.bias)[nc];
      if constexpr (Epi::kNumD >= 1) d0_v[o] = reinterpret_cast<const T*>(p.d0)[at];
      if constexpr (Epi::kNumD >= 2) d1_v[o] = reinterpret_cast<const T*>(p.d1)[at];
    }
  };

  f32x4 acc = {};
  // LOADS_A: of the rows of A that exist
  auto multiply_all = [&](auto loads_a) __attribute__((always_inline)) {
    constexpr int LOADS_A = decltype(loads_a)::value;
    auto issue = [&](int i, uint32_t at) __attribute__((always_inline)) {
      const int g = wave + i * NW;
      const int left = p.K - g * GROUP + (ELEM ? 1 : 0);  // elements of the group that exist (and the dword behind)
      const uint32_t k_at = (uint32_t)(g * GROUP) * 2u;
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int j = 0; j < (x == 0 ? LOADS_A : 4); ++j)
          rows_load_lds(ring + at + (uint32_t)(x * 4096 + j * 1024), piece[j] * 8 < left ? off[x][j] + k_at : kOobOffset, desc[x]);
    };
#pragma unroll
    for (int i = 0; i < NS; ++i)
      if (i < mine) issue(i, i * Tile::STAGE);
    read_epilogue();  // (the first wait, which counts them, takes in as many loads of the next group)
    uint32_t at = 0;
    // MORE: group i + NS is requested as soon as group i has been read (kAsk: if there is one)
    constexpr int kNo = 0, kYes = 1, kAsk = 2;
    auto multiply = [&](auto more, int i) __attribute__((always_inline)) {
      constexpr int MORE = decltype(more)::value;
      if (NS == 1 || MORE == kYes || i + NS - 1 < mine)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * (LOADS_A + 4)) : "memory");
      else  // (fewer than NS - 1 groups behind it)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      u32x4 f[2][4];
      uint32_t behind[2][4] = {};
      const uint32_t rd = ring + at + (uint32_t)(fr * 256);
      auto place = [&](int x, int c) __attribute__((always_inline)) { return rd + (uint32_t)(x * 4096 + (c ^ fr) * 16); };
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const bool none = ELEM && j == 3 && fq == 3;  // (the last piece is of the next group)
          rows_read16(f[x][j], none ? zeros : place(x, j * 4 + fq));
          if constexpr (ELEM != 0) rows_read4(behind[x][j], none ? zeros : place(x, (j * 4 + fq + 1) & 15));
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int x = 0; x < 2; ++x) rows_arrived(f[x][j], behind[x][j]);
      if (MORE == kYes || (MORE == kAsk && i + NS < mine)) issue(i + NS, at);
      at = at + Tile::STAGE == NS * Tile::STAGE ? 0 : at + Tile::STAGE;
      if constexpr (ELEM != 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            u32x4 r;
#pragma unroll
            for (int d = 0; d < 4; ++d) r[d] = __builtin_amdgcn_alignbit(d < 3 ? f[x][j][d < 3 ? d + 1 : 0] : behind[x][j], f[x][j][d], shift[x]);
            f[x][j] = r;
          }
      }
      // past the end of K: nothing of either operand
      const int g = wave + i * NW;
      if (MORE != kYes && g == groups - 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int left = p.K - g * GROUP - (j * 4 + fq) * 8;
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int d = 0; d < 4; ++d) f[x][j][d] &= left >= 2 * d + 2 ? 0xffffffffu : (left == 2 * d + 1 ? 0xffffu : 0u);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = Tr::mfma16(__builtin_bit_cast(vec8, f[1][j]), __builtin_bit_cast(vec8, f[0][j]), acc);
    };
    int i = 0;
    // (at odd elements in one loop: the shifts bound it and not the instructions of the cut, and two loops were 4 % slower above K = 4096)
    if constexpr (ELEM != 0) {
      for (; i < mine; ++i) multiply(std::integral_constant<int, kAsk>{}, i);
    } else {
      for (; i + NS < mine; ++i) multiply(std::integral_constant<int, kYes>{}, i);
      for (; i < mine; ++i) multiply(std::integral_constant<int, kNo>{}, i);
    }
  };
  if (rows_a <= 4)
    multiply_all(std::integral_constant<int, 1>{});
  else
    multiply_all(std::integral_constant<int, 4>{});

  // a lane holds columns 4 fq .. + 3 of row fr
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  float* const part = reinterpret_cast<float*>(smem_raw);  // [NW][16 rows of A][16 columns]
  *reinterpret_cast<f32x4*>(part + (wave * BM + fr) * BN + fq * 4) = acc;
  __syncthreads();
  float one = 1.0f;
  asm volatile("" : "+s"(one));  // (opaque to the optimizer: see to_float_plus)
  T* Cb = reinterpret_cast<T*>(p.c) + out_batch_offset(p, batch);
#pragma unroll
  for (int o = 0; o < OUTS; ++o) {
    const int m = out_m + o * (Tile::NT / BN);
    if (m < rows_a && out_n < rows_b) {
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += part[(w * BM + m) * BN + out_n];
      Cb[out_index<PERM>(p, m0 + m, n0 + out_n)] = epilogue1<Epi, T>(v, bias_v[o], d0_v[o], d1_v[o], one);
    }
  }
}

}  // namespace aitamd
