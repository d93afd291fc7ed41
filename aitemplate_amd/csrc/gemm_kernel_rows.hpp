// RCR GEMM for few rows of A: the weight matrix B streams through registers once, nothing is staged.
//
// Bound: HBM (or, for weights of a few hundred KiB, one trip to memory).  A launch cannot do without reading N x K
// weights; the M <= 16 MT rows of A are small and come from the caches.  A workgroup owns 16 columns of the output and
// its NW waves share K: wave w takes the 128-deep groups w, w + NW, ..., so that all of a short K is requested at once
// and of a long K every wave keeps up to 2 U groups (4 KiB of weights each) on their way.  v_mfma_f32_16x16x32 takes
// the 16 weight rows as one operand and 16 rows of A as the other, both as they come from memory (the padding rows of
// A cost matrix instructions only, and those have nothing else to do).  Which k an instruction multiplies is free as
// long as both operands agree: a lane's four pieces of a group are 64 consecutive bytes, so that the loads that touch
// a cache line follow each other at once (rows off 64-byte boundaries put two lines under every piece otherwise).
// The waves' partial tiles are added through LDS in wave order.
//
// Any K, pitch and alignment (ELEM; else dwords): rows are read in whole dwords, which rows at odd elements put
// together by shifts, as in the register-staged form of gemm_kernel_dma.hpp and for the same reasons.
//
// Measured: M=1 N=6912 K=8313 26.1 us = 4.4 TB/s (a large copy: 5.0), where the register-staged tiles take 40 and more;
// M=2 N=100 K=507 4.7 us (14.3 with element-wide loads).  From 17 rows on the 32-row tiles fetch A more cheaply.
#pragma once

#include "common.hpp"
#include "epilogue.hpp"
#include "gemm_kernel.hpp"

namespace aitamd {

// MT_: blocks of 16 rows of A; NW_: waves; U_: groups of 128 per half of the double-buffered pipeline
// ELEM_: rows at any element; 0: at dwords
template <int MT_, int NW_, int U_, int ELEM_>
struct GemmTileRows {
  static constexpr int ELEM = ELEM_;
  static constexpr int MT = MT_, NW = NW_, U = U_;
  static constexpr int BM = 16 * MT, BN = 16, BK = 128 * NW;  // (BK: what the waves take together)
  static constexpr int NT = NW * kWaveSize;
  static constexpr int KVEC = ELEM ? 1 : 2;
  static constexpr int kLdsBytes = NW * MT * 256 * 4;
  static constexpr int OUTS = (MT * 256 + NT - 1) / NT;  // outputs per thread
};

template <class T, class Tile, class Epi, bool PERM = false>
__global__ void __launch_bounds__(Tile::NT) gemm_rcr_rows_kernel(const GemmParams p) {
  using Tr = ElemTraits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int MT = Tile::MT, NW = Tile::NW, U = Tile::U;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  float* const part = reinterpret_cast<float*>(smem_raw);  // [NW][MT][16 rows of A][16 columns]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fq = lane >> 4;
  const int per_batch = p.tiles_m * p.tiles_n;
  const int batch = (int)blockIdx.x / per_batch;
  const int id = (int)blockIdx.x - batch * per_batch;
  const int tm = id / p.tiles_n;
  const int m0 = tm * Tile::BM, n0 = (id - tm * p.tiles_n) * Tile::BN;
  const int rows_a = (p.M - m0) < Tile::BM ? (p.M - m0) : Tile::BM;
  const int rows_b = (p.N - n0) < Tile::BN ? (p.N - n0) : Tile::BN;

  const T* Ab = reinterpret_cast<const T*>(p.a) + (int64_t)batch * p.sa + (int64_t)m0 * p.lda;
  const T* Bb = reinterpret_cast<const T*>(p.b) + (int64_t)batch * p.sb + (int64_t)n0 * p.ldb;
  const uint32_t odd_a = (uint32_t)(reinterpret_cast<uintptr_t>(Ab) & 3), odd_b = (uint32_t)(reinterpret_cast<uintptr_t>(Bb) & 3);
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(
      reinterpret_cast<const char*>(Ab) - odd_a, clamp_records(((((int64_t)rows_a - 1) * p.lda + p.K) * 2 + odd_a + 3) & ~3ll));
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(
      reinterpret_cast<const char*>(Bb) - odd_b, clamp_records(((((int64_t)rows_b - 1) * p.ldb + p.K) * 2 + odd_b + 3) & ~3ll));
  const uint32_t off_b = (uint32_t)(((int64_t)fr * p.ldb + fq * 32) * 2) + odd_b;
  uint32_t off_a[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) off_a[mt] = (uint32_t)(((int64_t)(mt * 16 + fr) * p.lda + fq * 32) * 2) + odd_a;

  // 64 consecutive bytes of a row: the dwords they start in and, for rows at odd elements, the one behind them
  struct Run {
    u32x4 v[4];
    uint32_t fifth;
  };
  auto read_run = [&](const __amdgpu_buffer_rsrc_t& r, uint32_t off, bool on) {
    Run x;
    const uint32_t at = on ? off & ~3u : kOobOffset;
#pragma unroll
    for (int j = 0; j < 4; ++j) x.v[j] = buffer_load_16B(r, at + j * 16);
    if constexpr (Tile::ELEM != 0) x.fifth = buffer_load_4B(r, at + 64);
    return x;
  };
  auto piece = [&](const Run& x, int j, uint32_t off) {
    u32x4 r = x.v[j];
    if constexpr (Tile::ELEM != 0) {
      const uint32_t shift = (off & 2u) * 8u;
#pragma unroll
      for (int d = 0; d < 4; ++d)
        r[d] = __builtin_amdgcn_alignbit(d < 3 ? x.v[j][d + 1] : (j < 3 ? x.v[j < 3 ? j + 1 : 3][0] : x.fifth), x.v[j][d], shift);
    }
    return r;
  };
  // K in groups of 128: groups 0 .. groups - 2 lie inside the rows; of the last one, whole or not, the wave whose turn
  // it is clears what lies past the end of K
  const int groups = (p.K + 127) / 128;
  const int mine = (groups - 1 - wave + NW - 1) / NW;  // whole groups of this wave
  const bool has_last = groups > 0 && (groups - 1) % NW == wave;
  const uint32_t last_at = (uint32_t)(groups - 1) * 256u;
  const int last_k = (groups - 1) * 128 + fq * 32;
  Run last_b, last_a[MT];
  if (has_last) {
    last_b = read_run(rb, off_b + last_at, last_k < p.K);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) last_a[mt] = read_run(ra, off_a[mt] + last_at, last_k < p.K);
  }

  Run wb[2][U], xa[2][U][MT];
  auto fetch = [&](auto half_c, int i0) {
    constexpr int H = decltype(half_c)::value;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t at = (uint32_t)(wave + (i0 + u) * NW) * 256u;
      wb[H][u] = read_run(rb, off_b + at, i0 + u < mine);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xa[H][u][mt] = read_run(ra, off_a[mt] + at, i0 + u < mine);
    }
  };
  f32x4 acc[MT] = {};
  auto multiply = [&](auto half_c) {
    constexpr int H = decltype(half_c)::value;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const vec8 w = __builtin_bit_cast(vec8, piece(wb[H][u], j, off_b));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[mt] = Tr::mfma16(w, __builtin_bit_cast(vec8, piece(xa[H][u][mt], j, off_a[mt])), acc[mt]);
      }
  };
  constexpr std::integral_constant<int, 0> h0{};
  constexpr std::integral_constant<int, 1> h1{};
  fetch(h0, 0);

  // what the epilogue reads, on its way beside the weights
  float bias_v[Tile::OUTS], d0_v[Tile::OUTS], d1_v[Tile::OUTS];
  const int64_t d_base = (int64_t)batch * p.sd;
#pragma unroll
  for (int o = 0; o < Tile::OUTS; ++o) {
    const int e = tid + o * Tile::NT;
    const int m = m0 + e / 16, n = n0 + e % 16;
    bias_v[o] = d0_v[o] = d1_v[o] = 0.0f;
    if (e < MT * 256 && m < p.M && n < p.N) {
      if constexpr (Epi::kHasBias) bias_v[o] = Tr::to_float(reinterpret_cast<const T*>(p.bias)[n]);
      if constexpr (Epi::kNumD >= 1) d0_v[o] = Tr::to_float(reinterpret_cast<const T*>(p.d0)[d_base + (int64_t)m * p.ldd + n]);
      if constexpr (Epi::kNumD >= 2) d1_v[o] = Tr::to_float(reinterpret_cast<const T*>(p.d1)[d_base + (int64_t)m * p.ldd + n]);
    }
  }

  for (int i0 = 0; i0 < mine; i0 += 2 * U) {
    fetch(h1, i0 + U);
    multiply(h0);
    fetch(h0, i0 + 2 * U);
    multiply(h1);
  }
  if (has_last) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int left = p.K - (last_k + j * 8);  // elements of the piece that exist
      auto cut = [&](u32x4 v) {
#pragma unroll
        for (int d = 0; d < 4; ++d) v[d] &= left >= 2 * d + 2 ? 0xffffffffu : (left == 2 * d + 1 ? 0xffffu : 0u);
        return __builtin_bit_cast(vec8, v);
      };
      const vec8 w = cut(piece(last_b, j, off_b));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = Tr::mfma16(w, cut(piece(last_a[mt], j, off_a[mt])), acc[mt]);
    }
  }

  // a lane holds columns 4 fq .. + 3 of row fr of every 16 x 16 block
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<f32x4*>(part + ((wave * MT + mt) * 16 + fr) * 16 + fq * 4) = acc[mt];
  __syncthreads();
  T* Cb = reinterpret_cast<T*>(p.c) + out_batch_offset(p, batch);
#pragma unroll
  for (int o = 0; o < Tile::OUTS; ++o) {
    const int e = tid + o * Tile::NT;
    const int m = m0 + e / 16, n = n0 + e % 16;
    if (e < MT * 256 && m < p.M && n < p.N) {
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += part[w * MT * 256 + e];
      Cb[out_index<PERM>(p, m, n)] = Tr::from_float(Epi::apply(v, bias_v[o], d0_v[o], d1_v[o]));
    }
  }
}

}  // namespace aitamd
