// Fused  out = softmax(scale * Q K^T) V  with the [B,M,O] -> [B/G, M, G, O] permute
// folded into the store (bmm_softmax_bmm_permute), gfx950.
//
// The score matrix never leaves the chip.  One wave owns 32 query rows and walks
// the keys/values in blocks of 32 (64 for the smallest head dims); a workgroup of 4 waves
// shares each 64- or 128-row K / V tile through LDS.  This kernel takes operands at any
// alignment through registers; attention_pipe.hpp has the one for whole 16-byte pieces.
//
//  * S^T = K Q^T is computed with v_mfma_f32_32x32x16 (K tile rows as the A
//    operand, the wave's Q rows - kept in registers for the whole kernel - as
//    the B operand).  In the accumulator layout of the transposed product a
//    lane holds 16 keys of ONE query row, so the online-softmax state (running
//    max, running sum, rescale factor) is one scalar per lane and the row
//    reductions are 15 in-lane ops plus a single v_permlane32_swap.
//  * The probabilities, rounded to the element type, are already laid out as the
//    B operand of the second MFMA  O^T = V^T P^T : no shuffle, no LDS round trip.
//  * V stays row-major [key][o] in LDS exactly as it sits in memory; the V^T
//    operand fragments are fetched with ds_read_b64_tr_b16 (LDS transpose read).
//  * head dims that are not MFMA multiples (40) are zero-padded inside the LDS
//    tiles only: K to 16*KS columns, V to 32*OT columns.
//
// Replaces DeviceBatchedGemmSoftmaxGemmPermute_Xdl_CShuffle as instantiated by
// the reference (python/aitemplate/utils/mk_ck_lib/gemm_operation.py:64,415-424;
// arguments python/aitemplate/backend/rocm/gemm/bmm_softmax_bmm_permute.py:84-110).
#pragma once

#include <type_traits>

#include "common.hpp"

#ifndef AITAMD_ATTN_KB
#define AITAMD_ATTN_KB(KS, OT) (((KS) + 2 * (OT)) <= 7 ? 2 : 1)
#endif

namespace aitamd {

struct AttnParams {
  const void* q;  // [B, M, K]
  const void* k;  // [B, N, K]
  const void* v;  // [B, N, O]
  void* out;      // [B / G, M, G, O]
  int32_t B, M, N, K, O, G;
  float scale_log2e;  // scale (already rounded to the element type) * log2(e)
  int32_t causal;
  // Optional, device memory, B / G entries: batch entry b only attends to its first kv_len[b / G] keys (clamped to
  // [0, N]); the later rows of K and V are never read.  Null: all N keys.
  const int32_t* kv_len;
  // Optional, same form: rows m >= q_len[b / G] of batch entry b are written as zeros, and a workgroup whose rows
  // all lie past that length visits no keys.
  const int32_t* q_len;
  // Non-zero: a NaN score counts as -inf (its key is left out of the row's softmax) instead of making the row NaN.
  int32_t nan_reset;
  // Non-zero (causal): the grid has half the query tiles, and a workgroup takes the i-th from the end and then the i-th.
  int32_t paired;
  // Set by the launcher of the pipelined kernel: the grid's extents (query tiles, batch entries), whether the entries are
  // dealt round the XCDs (a workgroup for every entry, fewer than 2^31), and the reciprocals of the tiles and of G.
  int32_t tiles, entries, dealt;
  Divisor by_tiles, by_heads;
};

// NW waves (32 query rows each) share the K / V tiles in two LDS stages
template <int KS_, int OT_>
struct AttnTile {
  static constexpr int KS = KS_;          // K padded to 16 * KS
  static constexpr int OT = OT_;          // O padded to 32 * OT
  static constexpr int KP = 16 * KS;
  static constexpr int OP = 32 * OT;
  static constexpr int NW = 4, NS = 2;
  static constexpr int BM = 32 * NW;      // query rows per workgroup
  static constexpr int BN = (16 * KS_ + 32 * OT_) <= 112 ? 128 : 64;  // keys per LDS tile: 128 while two workgroups still fit one CU's LDS
  static constexpr int NT = 64 * NW;
  static constexpr int K_PITCH = KP + 8;  // halves; keeps 16 consecutive rows on distinct banks
  // V rows carry no pad.  The transposing read fetches, per 32 lanes, 64 bytes of each of 4 consecutive rows; the
  // four pieces have to fall into four different quarters of the 64 banks.  Rows of 64 or 192 bytes do that as
  // they lie; rows of 128 or 256 bytes get the 64-byte pieces of a row exchanged by a row-dependent XOR.
  static constexpr int V_PITCH = OP;
  static constexpr int V_CR = OP / 8;                                             // 16-byte chunks per V row
  static constexpr int V_SWZ_GROUPS = (V_CR == 8 || V_CR == 16) ? V_CR / 4 : 1;  // 64-byte pieces exchanged
  static constexpr int V_SWZ_ROWS = V_CR == 8 ? 2 : 1;                            // rows per 256 bytes
  // chunk index -> chunk index ^ v_swz(row)
  static constexpr int v_swz(int row) { return 4 * ((row / V_SWZ_ROWS) % V_SWZ_GROUPS); }
  static constexpr int K_CHUNKS = BN * KP / 8;  // 16-byte chunks per tile (pads included)
  static constexpr int V_CHUNKS = BN * OP / 8;
  static constexpr int K_IT = (K_CHUNKS + NT - 1) / NT;
  static constexpr int V_IT = (V_CHUNKS + NT - 1) / NT;
  static constexpr int kLdsBytes = NS * BN * (K_PITCH + V_PITCH) * 2;
  static_assert(kLdsBytes <= 160 * 1024, "LDS budget");
};

// LDS transpose read: 4 x 16-bit per lane, gathered across the 16 lanes of a block (__restrict__: see tr_read16)
template <class T>
struct AttnVec;
template <>
struct AttnVec<f16> {
  typedef __fp16 raw4 __attribute__((__vector_size__(4 * sizeof(__fp16))));
  static AITAMD_DEVICE f16x4 tr_read(const f16* __restrict__ p) {
    const raw4 r = __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) raw4*)p);
    return __builtin_bit_cast(f16x4, r);
  }
  static AITAMD_DEVICE f16x4 tr_read(__attribute__((address_space(3))) const f16* __restrict__ p) {
    const raw4 r = __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) raw4*)p);
    return __builtin_bit_cast(f16x4, r);
  }
};
template <>
struct AttnVec<bf16> {
  typedef __bf16 raw4 __attribute__((__vector_size__(4 * sizeof(__bf16))));
  static AITAMD_DEVICE bf16x4 tr_read(const bf16* __restrict__ p) {
    const raw4 r = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) raw4*)p);
    return __builtin_bit_cast(bf16x4, r);
  }
  static AITAMD_DEVICE bf16x4 tr_read(__attribute__((address_space(3))) const bf16* __restrict__ p) {
    const raw4 r = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) raw4*)p);
    return __builtin_bit_cast(bf16x4, r);
  }
};

// acc + the 8 elements of v: four v_dot2 against (1, 1) on the packed pairs as they lie in the registers
AITAMD_DEVICE float add_elements(f16x8 v, float acc) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  struct Quads {
    h2 q[4];
  };
  const Quads u = __builtin_bit_cast(Quads, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_fdot2(u.q[i], h2{(f16)1.0f, (f16)1.0f}, acc, false);
  return acc;
}
AITAMD_DEVICE float add_elements(bf16x8 v, float acc) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  struct Quads {
    b2 q[4];
  };
  const Quads u = __builtin_bit_cast(Quads, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_fdot2_f32_bf16(u.q[i], b2{(bf16)1.0f, (bf16)1.0f}, acc, false);
  return acc;
}

AITAMD_DEVICE float max_across_halves(float x) {
  // lane l and lane l^32 hold the two halves of one query row
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
AITAMD_DEVICE float sum_across_halves(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The row sum (of one lane's half of the keys) up to which probabilities may be taken against an old reference point;
// beyond it, and at NaN, a tile is done again in the full form.  The accumulators hold the sum times the values, so
// they stay finite for values up to 2^87; a bound near the largest float, which only the probabilities of bf16 get to
// without being infinite, let the product with values above 1 overflow.  The full form itself lets a row's sum grow to
// 2^8 a key (kLazyLog2), 2^39 for the most keys there can be, which therefore does not trip it.
constexpr float kMaxRowSum = 0x1p40f;

template <int N>
AITAMD_DEVICE void attn_wait_vmcnt() {
  // s_waitcnt simm16: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt_hi[15:14]; only vmcnt is waited for
  constexpr int imm = (N & 0xf) | ((N >> 4) << 14) | (0x7 << 4) | (0xf << 8);
  __builtin_amdgcn_s_waitcnt(imm);
}
// VEC: K and O are multiples of 8 and all base pointers 16-byte aligned -> 128-bit
// loads; otherwise elements are gathered one by one (slow, any shape).
template <class T, class Tile, bool VEC>
__global__ void __launch_bounds__(Tile::NT, 2) attention_kernel(const AttnParams p) {
  constexpr int NS = Tile::NS;
  using Tr = ElemTraits<T>;
  using vec8 = typename Tr::vec8;
  using vec4 = typename Tr::vec4;
  constexpr int KS = Tile::KS, OT = Tile::OT, KP = Tile::KP, OP = Tile::OP;
  constexpr int BN = Tile::BN, KPI = Tile::K_PITCH, VPI = Tile::V_PITCH;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  T* const sK = reinterpret_cast<T*>(smem_raw);  // [NS][BN][K_PITCH]
  T* const sV = sK + NS * BN * KPI;              // [NS][BN][V_PITCH]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;  // which 32 query rows
  const int r32 = lane & 31;
  const int h = lane >> 5;
  const int m0 = blockIdx.x * Tile::BM;
  for (int b = blockIdx.y; b < p.B; b += gridDim.y) {
    const int q_row = m0 + wave * 32 + r32;  // this lane's query row
    const T* Qb = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.M * p.K;
    const T* Kb = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.N * p.K;
    const T* Vb = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.N * p.O;
    // keys of this batch entry (uniform over the workgroup)
    int N = p.N;
    if (p.kv_len != nullptr) {
      const int len = __builtin_amdgcn_readfirstlane(p.kv_len[b / p.G]);
      N = len < 0 ? 0 : (len < N ? len : N);
    }
    int m_rows = p.M;
    if (p.q_len != nullptr) {
      const int len = __builtin_amdgcn_readfirstlane(p.q_len[b / p.G]);
      m_rows = len < 0 ? 0 : (len < m_rows ? len : m_rows);
      if (m0 >= m_rows) N = 0;  // nothing but padding rows here: no keys, zeros out
    }

    // ---- Q fragments (B operand of S^T = K Q^T): lane (q = r32, k = 16 ks + 8 h + j)
    vec8 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int k0 = ks * 16 + h * 8;
      vec8 v = {};
      if (q_row < p.M) {
        if (VEC) {
          if (k0 < p.K) v = *reinterpret_cast<const vec8*>(Qb + (int64_t)q_row * p.K + k0);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (k0 + j < p.K) v[j] = Qb[(int64_t)q_row * p.K + k0 + j];
        }
      }
      // a negative scale changes sides: (-Q) K^T with |scale| gives the same scaled scores, and the
      // softmax below only ever sees a positive scale (negation is exact)
      if (p.scale_log2e < 0.0f) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = -v[j];
      }
      qf[ks] = v;
    }

    // ---- tile loaders: global -> registers -> LDS, zero-filled past N / K / O
    u32x4 kreg[Tile::K_IT], vreg[Tile::V_IT];
    auto gather = [&](const T* base, int row, int col, int rows, int cols) -> u32x4 {
      union {
        u32x4 v;
        T e[8];
      } u;
      u.v = u32x4{0, 0, 0, 0};
      if (row < rows) {
        if (VEC) {
          if (col < cols) u.v = *reinterpret_cast<const u32x4*>(base + (int64_t)row * cols + col);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (col + j < cols) u.e[j] = base[(int64_t)row * cols + col + j];
        }
      }
      return u.v;
    };
    auto load_tiles = [&](int n0) {
#pragma unroll
      for (int i = 0; i < Tile::K_IT; ++i) {
        const int c = tid + i * Tile::NT;
        const int row = c / (KP / 8), col = (c % (KP / 8)) * 8;
        kreg[i] = (c < Tile::K_CHUNKS) ? gather(Kb, n0 + row, col, N, p.K) : u32x4{0, 0, 0, 0};
      }
#pragma unroll
      for (int i = 0; i < Tile::V_IT; ++i) {
        const int c = tid + i * Tile::NT;
        const int row = c / (OP / 8), col = (c % (OP / 8)) * 8;
        vreg[i] = (c < Tile::V_CHUNKS) ? gather(Vb, n0 + row, col, N, p.O) : u32x4{0, 0, 0, 0};
      }
    };
    auto store_tiles = [&](int stage) {
      T* dK = sK + stage * BN * KPI;
      T* dV = sV + stage * BN * VPI;
#pragma unroll
      for (int i = 0; i < Tile::K_IT; ++i) {
        const int c = tid + i * Tile::NT;
        const int row = c / (KP / 8), col = (c % (KP / 8)) * 8;
        if (c < Tile::K_CHUNKS) *reinterpret_cast<u32x4*>(dK + row * KPI + col) = kreg[i];
      }
#pragma unroll
      for (int i = 0; i < Tile::V_IT; ++i) {
        const int c = tid + i * Tile::NT;
        const int row = c / (OP / 8), col = (c % (OP / 8)) * 8;
        if (c < Tile::V_CHUNKS) *reinterpret_cast<u32x4*>(dV + row * VPI + (col ^ (Tile::v_swz(row) * 8))) = vreg[i];
      }
    };

    const int wave_u = __builtin_amdgcn_readfirstlane(wave);

    // keys this workgroup has to visit (causal: nothing right of the last query row)
    int n_end = N;
    if (p.causal) {
      const int last = m0 + Tile::BM;
      n_end = last < n_end ? last : n_end;
    }
    const int n_tiles = (n_end + BN - 1) / BN;

    f32x16 oacc[OT];
#pragma unroll
    for (int ot = 0; ot < OT; ++ot)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[ot][e] = 0.0f;
    // running maximum of the raw scores of this lane's row (of the negated scores when the scale is
    // negative: see the Q fragments)
    const float c = __builtin_fabsf(p.scale_log2e);
    float m_run = -INFINITY;
    float l_run = 0.0f;       // running sum over this lane's half of the keys
    bool ref_ok = false;      // (wave-uniform) every row of the wave has a finite reference point

    if (n_tiles > 0) {
      load_tiles(0);
      store_tiles(0);
    }
    __syncthreads();

    // source-lane address pattern of the LDS transpose read (see file header):
    // 16-lane block = one 4-key x 16-column patch; lane i of the block points at
    // key i/4, columns 4*(i%4)..+3 of the patch.
    const int tr_i = lane & 15;
    const int tr_row = tr_i >> 2;
    const int tr_col = ((lane >> 4) & 1) * 16 + (tr_i & 3) * 4;
    // every row a lane reads is its tr_row plus a multiple of 4: one swizzle value per lane
    const int tr_swz = Tile::v_swz(tr_row) * 8;

    // 32-key sub-blocks per softmax step: two for head dims up to 48, which halves the per-step work (exchange
    // across halves, rescale test, branches) per key: 3.7 % faster at head dim 40; at 64 the 16 extra
    // registers cost a resident workgroup and it measures equal, so one there
    constexpr int KB = AITAMD_ATTN_KB(KS, OT);
    static_assert(BN % (32 * KB) == 0, "a tile is whole blocks");
    int cur = 0;
    for (int t = 0; t < n_tiles; ++t) {
      const bool has_next = (t + 1) < n_tiles;
      if (has_next) load_tiles((t + 1) * BN);
      const T* cK = sK + cur * BN * KPI;
      const T* cV = sV + cur * BN * VPI;
      // The lane's LDS addresses of the tile, one per operand (and per 32-column block of V, whose swizzle sits
      // in the column bits), taken once per tile and made opaque: every fragment read of the tile is then that
      // register plus an immediate offset.  Left to itself the compiler re-adds stage base, lane offset and block
      // offset in front of every read (22 vector instructions per 64 keys).
      typedef __attribute__((address_space(3))) const T lds_T;
      lds_T* k_lane = (lds_T*)(cK + r32 * KPI + h * 8);
      asm volatile("" : "+v"(k_lane));
      lds_T* v_lane[OT];
#pragma unroll
      for (int ot = 0; ot < OT; ++ot) {
        v_lane[ot] = (lds_T*)(cV + (h * 4 + tr_row) * VPI + ((ot * 32) ^ tr_swz) + tr_col);
        asm volatile("" : "+v"(v_lane[ot]));
      }

#pragma unroll
      for (int blk = 0; blk < BN / (32 * KB); ++blk) {
        const int nb = t * BN + blk * 32 * KB;  // first key of this block of KB x 32 keys
        // ---- S^T sub-blocks: rows = keys, columns = this wave's 32 query rows
        // (issuing the next block's product ahead of this block's softmax was measured: no gain at
        // head dim 40 and a quarter slower at head dim 64, where the extra live accumulator costs more)
        f32x16 s[KB];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
          for (int e = 0; e < 16; ++e) s[kb][e] = 0.0f;
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            typedef __attribute__((address_space(3))) const vec8 lds_vec8;
            const vec8 kf = *(lds_vec8*)(k_lane + (blk * KB + kb) * 32 * KPI + ks * 16);
            s[kb] = Tr::mfma32(kf, qf[ks], s[kb]);
          }
        }
        // lane holds keys nb + 32 kb + 8 g + 4 h + r (element 4 g + r of sub-block kb) of query row q_row.
        // The running maximum is kept on the raw scores and the scale is folded into the exponent:
        // p = exp2(s * c - m * c) is one FMA and one v_exp per score (c > 0: a negative scale was moved into
        // the Q fragments).  Only blocks that reach past N or touch the causal diagonal pay for masking; the
        // test is wave-uniform, so it costs one scalar branch per block.
        const bool need_mask = (nb + 32 * KB > N) || (p.causal && nb + 32 * KB - 1 > m0 + wave_u * 32);
        float alpha = 1.0f;
        vec8 pf[2 * KB];  // P^T fragments of the block's 16-key steps
        auto softmax_block = [&](auto masked_tag, auto nan_tag) {
          constexpr bool MASKED = decltype(masked_tag)::value;
          constexpr bool NAN_RESET = decltype(nan_tag)::value;  // (implies MASKED)
          bool dead[KB][16];
          if constexpr (MASKED) {
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
              for (int e = 0; e < 16; ++e) {
                const int n = nb + kb * 32 + (e >> 2) * 8 + h * 4 + (e & 3);
                dead[kb][e] = (n >= N) || (p.causal && n > q_row) || (NAN_RESET && s[kb][e] != s[kb][e]);
              }
          }
          float text = -INFINITY;
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int e = 0; e < 16; ++e) text = fmaxf(text, (MASKED && dead[kb][e]) ? -INFINITY : s[kb][e]);
          text = max_across_halves(text);
          const float m_cand = fmaxf(m_run, text);
          // The reference point of the exponent moves only when the row maximum has grown by more than
          // kLazyLog2 binary orders since it was last taken: until then p = exp2(s c - m c) may exceed 1 (by at
          // most 2^kLazyLog2, harmless in fp32 sums and in the fp16 / bf16 probabilities) and the accumulators
          // need no rescaling.  With random scores some row of a wave sets a new maximum in most blocks, so
          // rescaling on every change costs 2 multiplies per score; this way it is rare.
          constexpr float kLazyLog2 = 8.0f;
          const float drift = (m_run - m_cand) * c;  // <= 0; -inf (or NaN for inf - inf) on the first live block
          const bool move = !(drift >= -kLazyLog2);
          const float m_new = move ? m_cand : m_run;
          const float m_safe = __builtin_isinf(m_new) ? 0.0f : m_new;  // every key so far masked
          alpha = !move ? 1.0f : (__builtin_isinf(m_run) ? 0.0f : __builtin_amdgcn_exp2f(drift));
          const float mc = -m_safe * c;
          // the probabilities are rounded to the element type at once (the second product takes them so) and the
          // row sum adds the rounded values, two per instruction
          l_run *= alpha;
#pragma unroll
          for (int st = 0; st < 2 * KB; ++st) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const int kb = st >> 1, e = (st & 1) * 8 + j;
              pf[st][j] = Tr::from_float(
                  (MASKED && dead[kb][e]) ? 0.0f : __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][e], c, mc)));
            }
            l_run = add_elements(pf[st], l_run);
          }
          m_run = m_new;
        };
        const float m_before = m_run, l_before = l_run;
        // Fast form of an unmasked block: no row maximum at all.  The probabilities are taken against the reference
        // point the row already has, p = exp2((s - m) c); that is exact whatever m is, as long as neither p nor its
        // product with the values leaves its type's range, and a row sum that is NaN or beyond kMaxRowSum has the block
        // redone below in the full form (maximum, moved reference point, rescaled accumulators).  After a row's
        // first block - always the full form: there is no reference point yet - that takes a score 16 binary orders
        // above everything the row has seen (fp16; some 36 for bf16), so nearly every block saves the
        // maximum's 16 three-way compares, the exchange across the wave's halves and the bookkeeping of the
        // reference point: 96 instead of 128 vector instructions per 64 keys.
        bool full = need_mask || !ref_ok;
        if (!full) {
          const float mc = -m_run * c;
#pragma unroll
          for (int st = 0; st < 2 * KB; ++st) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const int kb = st >> 1, e = (st & 1) * 8 + j;
              pf[st][j] = Tr::from_float(__builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][e], c, mc)));
            }
            l_run = add_elements(pf[st], l_run);
          }
          if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(l_run <= kMaxRowSum)) != 0, 0)) {
            l_run = l_before;
            full = true;
          }
        }
        if (full) {
          if (need_mask)
            softmax_block(std::true_type{}, std::false_type{});
          else
            softmax_block(std::false_type{}, std::false_type{});
          ref_ok = __builtin_amdgcn_ballot_w64(__builtin_isinf(m_run)) == 0;
        }
        // A NaN score (a NaN in Q or in a K row) counts as -inf, i.e. its key is left out, as in the reference, whose
        // kernel applies ScaleAndResetNaNToMinusInfinity to the scores
        // (python/aitemplate/backend/rocm/gemm/bmm_softmax_bmm_permute.py:106, bmm_softmax_bmm.py:99).  The running
        // maximum ignores NaNs as it is (fmaxf), and a NaN probability shows in the lane's row sum: the block is redone
        // with those keys masked.  One compare and one scalar branch per block where there is none.  (mem_eff_attention
        // runs without the reset: the reference's kernel for it only scales.)
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(l_run != l_run) != 0, 0) && p.nan_reset) {
          m_run = m_before;
          l_run = l_before;
          softmax_block(std::true_type{}, std::true_type{});
          ref_ok = __builtin_amdgcn_ballot_w64(__builtin_isinf(m_run)) == 0;
        }
        if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
          for (int ot = 0; ot < OT; ++ot)
#pragma unroll
            for (int e = 0; e < 16; ++e) oacc[ot][e] *= alpha;
        }
        // ---- O^T += V^T P^T over the block's 16-key steps
#pragma unroll
        for (int st = 0; st < 2 * KB; ++st) {
#pragma unroll
          for (int ot = 0; ot < OT; ++ot) {
            lds_T* vb = v_lane[ot] + (blk * KB * 32 + st * 16) * VPI;
            const vec4 lo = AttnVec<T>::tr_read(vb);
            const vec4 hi = AttnVec<T>::tr_read(vb + 8 * VPI);
            vec8 vf;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              vf[j] = lo[j];
              vf[4 + j] = hi[j];
            }
            oacc[ot] = Tr::mfma32(vf, pf[st], oacc[ot]);
          }
        }
      }

      if (has_next) store_tiles(cur ^ 1);
      __syncthreads();
      cur ^= 1;
    }

    // ---- normalise and store permuted: out[b / G][m][b % G][o]
    const float l_tot = sum_across_halves(l_run);
    const float inv = (l_tot > 0.0f && q_row < m_rows) ? 1.0f / l_tot : 0.0f;
    if (q_row < p.M) {
      T* orow = reinterpret_cast<T*>(p.out) + (((int64_t)(b / p.G) * p.M + q_row) * p.G + (b % p.G)) * p.O;
      const bool vec_ok = ((p.O & 3) == 0) && ((reinterpret_cast<uintptr_t>(p.out) & 7) == 0);
#pragma unroll
      for (int ot = 0; ot < OT; ++ot)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int o = ot * 32 + g * 8 + h * 4;
          if (o >= p.O) continue;
          if (vec_ok) {
            vec4 ov;
#pragma unroll
            for (int j = 0; j < 4; ++j) ov[j] = Tr::from_float(oacc[ot][g * 4 + j] * inv);
            *reinterpret_cast<vec4*>(orow + o) = ov;
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (o + j < p.O) orow[o + j] = Tr::from_float(oacc[ot][g * 4 + j] * inv);
          }
        }
    }
    __builtin_amdgcn_s_barrier();  // every wave has left the stages that the next iteration refills
  }
}

}  // namespace aitamd
