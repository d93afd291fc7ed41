// Fused  out = softmax(scale * Q K^T) V  with the [B,M,O] -> [B/G, M, G, O] permute folded into the store, for head
// dims in whole 16-byte pieces: the pipelined form (attention_kernel.hpp has the form for all other operands and
// describes the score product in transposed form, which this one shares).
//
// A wave owns QB x 32 query rows and takes one tile of BN = 32 KB keys per iteration; its workgroup's K and V tiles go
// straight from memory to LDS, D tiles ahead.  The second product runs one tile behind the first: an iteration is
//     S(t) = K(t) Q^T;   O += V(t-1) P(t-1)  and, between its matrix instructions,  P(t) = exp2(c S(t) - c m)
// in one straight line, so the matrix unit works on tile t-1 while the exponentials of tile t are taken, and nothing
// of the tile is waited for but its scores.  The V ring keeps one tile more than the K ring for it.
//  * P against the reference point m the row already has (exact whatever m is, as long as neither P nor its product with
//    the values leaves its type's range; a row sum that is NaN or beyond kMaxRowSum has the tile done again in the full form).
//  * full form: a row's first tile, tiles that reach past the keys or over the causal diagonal, NaN scores, and rows
//    whose maximum has grown out of range: masks, maximum, moved reference point, rescaled accumulators.
//  * NG groups of NW waves take alternate parts of a tile of NG x BN keys and merge at the end: for grids that leave
//    CUs idle.
//
// What bounds it: at head dims 64 and below the exponentials and the conversions around them (a quarter-rate
// instruction per score against 1/8 of a matrix instruction per 64 of them), at 128 and above the matrix unit and the
// LDS reads of K and V that feed it.  Doing one product after the other, as the staged form does, had the matrix unit
// wait for each tile's exponentials and the wave wait for every fragment it read.  us, fp16, before -> now:
//   1 x 16 x 8192^2, d 64          327 -> 288    2 x 16 x 4096^2, d 128, bf16           311 -> 262
//   4 x 8 x 4096^2, d 80           229 -> 212    2 x 16 x 4096^2, d 128, bf16, causal   176 -> 142
//   2 x 8 x 1024^2, d 160           43 -> 31     64 x 12 x 384^2, d 64, mixed lengths    45 -> 40
//   and short calls (a few heads of up to 128 keys), that a launch and one tile's latency bound: 7 to 13 -> 4 to 8.
// What comes ahead of the first tile counts for those: 345 instructions and four trips to memory one after the other
// (arguments, grid, lengths, Q) until coordinates came without divisions and Q was asked for ahead of the lengths, 227 and
// two: 768 x 64^2 with lengths 7.8 -> 7.3, 88 x 195^2 at d 128 10.3 -> 9.9, 144 x 41^2 4.2 -> 4.0, 16 x 200^2 4.9 -> 4.7.
// Tried and not kept: the scores one tile further ahead (S twice in registers: slower at every head dim), one more
// stage in both rings (nothing), no tile asked for past the last (a branch in the loop: 2 % slower), row sums by a 4x4x4
// matrix instruction (3 % slower; no sums at all are 2 % faster), K fragments read a tile ahead (even, spills at 128), three
// or four workgroups per CU at head dim 80 and above (spills), 8 waves on one K / V tile (head dim 80 5 % faster, 128
// even, 64 slower).
#pragma once

#include "attention_kernel.hpp"

namespace aitamd {

template <int KS_, int OT_, int KB_, int NW_, int QB_, int NG_, int D_, int OCC_>
struct AttnPipe {
  static constexpr int KS = KS_, OT = OT_, KB = KB_, NW = NW_, QB = QB_, NG = NG_, D = D_, OCC = OCC_;
  static constexpr int KP = 16 * KS, OP = 32 * OT;
  static constexpr int BN = 32 * KB, BNT = BN * NG;  // keys of a tile per group and in all
  static constexpr int BM = 32 * QB * NW;
  static constexpr int NWT = NW * NG, NT = 64 * NWT;
  static constexpr int K_PITCH = KP + 8;  // halves; keeps 16 consecutive rows on distinct banks
  static constexpr int V_PITCH = OP;      // (swizzled: see AttnTile)
  static constexpr int KC1 = K_PITCH / 8, VC1 = OP / 8;  // 16-byte pieces per LDS row
  static constexpr int KL = (BNT * KC1 + 63) / 64, VL = (BNT * VC1 + 63) / 64;  // wave-loads per tile
  static constexpr int K_IT = (KL + NWT - 1) / NWT, V_IT = (VL + NWT - 1) / NWT;
  static constexpr int NK = D + 1, NV = D + 2;
  static constexpr int K_STAGE = KL * 512, V_STAGE = VL * 512;  // elements
  static constexpr int O_PITCH = OP + 8;
  static constexpr int kRing = (NK * K_STAGE + NV * V_STAGE) * 2;
  static constexpr int kStrips = NW * 32 * O_PITCH * 2;
  static constexpr int kMerge = NG > 1 ? (16 * OT + 2) * QB * NW * 64 * 4 : 0;
  static constexpr int kLdsBytes = kRing > kStrips ? (kRing > kMerge ? kRing : kMerge) : (kStrips > kMerge ? kStrips : kMerge);
  static constexpr int v_swz(int row) { return AttnTile<KS, OT>::v_swz(row); }
  static_assert(kLdsBytes <= 160 * 1024, "LDS budget");
};

template <class T, class Tile>
__global__ void __launch_bounds__(Tile::NT, Tile::OCC) attention_pipe_kernel(const AttnParams p) {
  using Tr = ElemTraits<T>;
  using vec8 = typename Tr::vec8;
  using vec4 = typename Tr::vec4;
  typedef __attribute__((address_space(3))) void lds_void;
  typedef __attribute__((address_space(3))) const T lds_T;
  typedef __attribute__((address_space(3))) const vec8 lds_vec8;
  constexpr int KS = Tile::KS, OT = Tile::OT, KB = Tile::KB, QB = Tile::QB, NW = Tile::NW, NG = Tile::NG, NWT = Tile::NWT;
  constexpr int BN = Tile::BN, BNT = Tile::BNT, KPI = Tile::K_PITCH, VPI = Tile::V_PITCH, NK = Tile::NK, NV = Tile::NV, D = Tile::D;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  T* const sK = reinterpret_cast<T*>(smem_raw);
  T* const sV = sK + NK * Tile::K_STAGE;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave_all / NW, wave = wave_all % NW;
  const int r32 = lane & 31, h = lane >> 5;

  // Workgroup -> (query tile, batch entry).  The hardware deals consecutive workgroup ids round-robin over the
  // 8 XCDs, each with its own L2; XCD x works through the batch entries x, x + 8, x + 16, ... one after the other, so
  // the workgroups that stream the same K / V share one L2 and long and short sequences are spread over the XCDs.  The
  // up to seven entries that are left over go round the XCDs tile by tile.  Causal: the longest rows first.
  // (the arguments with one wait and coordinates without divisions: see fetch_arguments and Divisor)
  asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.B), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.O), "s"(p.G), "s"(p.causal), "s"(p.kv_len),
               "s"(p.q_len), "s"(p.tiles), "s"(p.dealt), "s"(p.by_tiles.mul), "s"(p.by_tiles.shift), "s"(p.by_heads.mul), "s"(p.by_heads.shift));
  int bx = blockIdx.x, by = blockIdx.y;
  if (p.dealt) {
    const int id = bx + p.tiles * by;
    const int even = p.B & ~(kNumXcd - 1);
    if (id < even * p.tiles) {
      const int slot = (int)((uint32_t)id / kNumXcd), entry = quotient(slot, p.by_tiles);
      by = entry * kNumXcd + (int)((uint32_t)id % kNumXcd);
      bx = slot - entry * p.tiles;
    }
    if (p.causal) bx = p.tiles - 1 - bx;
  }
  const int m_tiles = (p.M + Tile::BM - 1) / Tile::BM;
  const int first_tile = p.paired ? m_tiles - 1 - (p.tiles - 1 - bx) : bx;
  const int passes = p.paired && 2 * first_tile != m_tiles - 1 ? 2 : 1;

  // lane offsets of the tile loads: load i of a wave fills 1 KiB block wave_all + NWT * i of the K (V) stage
  uint32_t k_off[Tile::K_IT], v_off[Tile::V_IT];
#pragma unroll
  for (int i = 0; i < Tile::K_IT; ++i) {
    const int idx = (wave_all + NWT * i) * 64 + lane, row = idx / Tile::KC1, ch = idx - row * Tile::KC1;
    k_off[i] = (ch * 8 < p.K && row < BNT) ? (uint32_t)((row * p.K + ch * 8) * 2) : kOobOffset;
  }
#pragma unroll
  for (int i = 0; i < Tile::V_IT; ++i) {
    const int idx = (wave_all + NWT * i) * 64 + lane, row = idx / Tile::VC1;
    const int ch = (idx - row * Tile::VC1) ^ Tile::v_swz(row);
    v_off[i] = (ch * 8 < p.O && row < BNT) ? (uint32_t)((row * p.O + ch * 8) * 2) : kOobOffset;
  }
  // LDS offsets of the fragment reads
  const int k_rd = (grp * BN + r32) * KPI + h * 8;
  const int tr_row = (lane & 15) >> 2;
  const int tr_col = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
  const int tr_swz = Tile::v_swz(tr_row) * 8;
  int v_rd[OT];
#pragma unroll
  for (int ot = 0; ot < OT; ++ot) v_rd[ot] = (grp * BN + h * 4 + tr_row) * VPI + ((ot * 32) ^ tr_swz) + tr_col;

  // (a scale of zero counts as one that makes every score the same)
  const float c = fmaxf(__builtin_fabsf(p.scale_log2e), 1e-37f);
  const uint32_t flip = p.scale_log2e < 0.0f ? 0x80008000u : 0u;  // a negative scale changes sides: (-Q) K^T, exact

  for (int b = by, pass = 0; b < p.B; pass = pass + 1 < passes ? pass + 1 : 0, b += pass == 0 ? p.entries : 0) {
    const int m0 = (pass == 0 ? first_tile : m_tiles - 1 - first_tile) * Tile::BM;
    const int w0 = m0 + wave * 32 * QB;  // first row of this wave
    // Q fragments (B operand of S^T = K Q^T): lane (q = r32, k = 16 ks + 8 h + j).  Asked for first: nothing about them
    // depends on the entry's lengths, which are a trip to memory of their own.
    u32x4 raw[QB][KS];
    {
      const int rows = p.M - m0 < Tile::BM ? p.M - m0 : Tile::BM;
      const __amdgpu_buffer_rsrc_t rq = make_rsrc(
          reinterpret_cast<const T*>(p.q) + ((int64_t)b * p.M + m0) * p.K, rows > 0 ? (uint32_t)(rows * p.K * 2) : 0u);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int k0 = ks * 16 + h * 8;
          raw[qb][ks] = buffer_load_16B(rq, k0 < p.K ? (uint32_t)((((wave * QB + qb) * 32 + r32) * p.K + k0) * 2) : kOobOffset);
        }
    }
    const int seq = quotient(b, p.by_heads);
    // Through the scalar cache: nothing writes them while this runs.  A scalar load takes an address without its low two
    // bits, and the lengths may lie at any byte: the dwords of the first and the last byte of one, which are the same where
    // it is whole.  (Behind the asm, so that nothing of the address is held in registers from one entry to the next.)
    auto lengths = [&](const int32_t* of) __attribute__((always_inline)) {
      typedef const __attribute__((address_space(4))) uint32_t* scalar_ptr;
      uintptr_t at = reinterpret_cast<uintptr_t>(of) + 4 * (uintptr_t)(uint32_t)seq;
      asm("" : "+s"(at));
      const uint64_t lo = *(scalar_ptr)(at & ~(uintptr_t)3), hi = *(scalar_ptr)((at + 3) & ~(uintptr_t)3);
      return __builtin_amdgcn_readfirstlane((int)((hi << 32 | lo) >> (8 * (at & 3))));
    };
    int N = p.N;
    if (p.kv_len != nullptr) {
      const int len = lengths(p.kv_len);
      N = len < 0 ? 0 : (len < N ? len : N);
    }
    int m_rows = p.M;
    if (p.q_len != nullptr) {
      const int len = lengths(p.q_len);
      m_rows = len < 0 ? 0 : (len < m_rows ? len : m_rows);
      if (m0 >= m_rows) N = 0;  // nothing but padding rows here: no keys, zeros out
    }
    // keys this workgroup has to visit (causal: nothing right of the last query row)
    const int n_end = p.causal && m0 + Tile::BM < N ? m0 + Tile::BM : N;
    const int n_tiles = (n_end + BNT - 1) / BNT;
    // keys that some row, and that every row of this wave sees
    const int w_some = p.causal && w0 + 32 * QB < N ? w0 + 32 * QB : N;
    const int w_every = p.causal && w0 + 1 < N ? w0 + 1 : N;

    const __amdgpu_buffer_rsrc_t rk =
        make_rsrc(reinterpret_cast<const T*>(p.k) + (int64_t)b * p.N * p.K, (uint32_t)((int64_t)n_end * p.K * 2));
    const __amdgpu_buffer_rsrc_t rv =
        make_rsrc(reinterpret_cast<const T*>(p.v) + (int64_t)b * p.N * p.O, (uint32_t)((int64_t)n_end * p.O * 2));
    int k_in = 0, v_in = 0;  // stages that the next loads go to
    auto issue = [&](int t) {
      const uint32_t k_step = (uint32_t)(t * BNT * p.K * 2), v_step = (uint32_t)(t * BNT * p.O * 2);
      T* dK = sK + k_in * Tile::K_STAGE + wave_all * 512;
      T* dV = sV + v_in * Tile::V_STAGE + wave_all * 512;
#pragma unroll
      for (int i = 0; i < Tile::K_IT; ++i) {
        if ((i + 1) * NWT > Tile::KL && wave_all + i * NWT >= Tile::KL) continue;
        const uint32_t off = k_off[i] + k_step;  // (an out-of-range one stays out of range)
        T* dst = dK + i * NWT * 512;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_void*)dst, 16, off, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < Tile::V_IT; ++i) {
        if ((i + 1) * NWT > Tile::VL && wave_all + i * NWT >= Tile::VL) continue;
        const uint32_t off = v_off[i] + v_step;
        T* dst = dV + i * NWT * 512;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_void*)dst, 16, off, 0, 0, 0);
      }
      k_in = k_in + 1 == NK ? 0 : k_in + 1;
      v_in = v_in + 1 == NV ? 0 : v_in + 1;
    };
    if (n_tiles > 0) {
#pragma unroll
      for (int t = 0; t < D; ++t) issue(t);
    }
    // (used here, so that Q is waited for ahead of the loop and the tiles behind it are not)
    vec8 qf[QB][KS];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int d = 0; d < 4; ++d) raw[qb][ks][d] ^= flip;
        qf[qb][ks] = __builtin_bit_cast(vec8, raw[qb][ks]);
      }

    f32x16 oacc[QB][OT];
    float m_run[QB], l_run[QB];
    vec8 pf[QB][2 * KB];  // P^T fragments of the tile whose second product is due
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
      for (int ot = 0; ot < OT; ++ot)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[qb][ot][e] = 0.0f;
      m_run[qb] = -INFINITY;
      l_run[qb] = 0.0f;
    }
    bool due = false;     // (wave-uniform) pf holds a tile's probabilities
    bool ref_ok = false;  // (wave-uniform) every row of the wave has a finite reference point
    int k_at = 0, v_at = 0;  // stages of K(t) and V(t - 1)

    auto read_v = [&](lds_T* base, int st, int ot) {
      const vec4 lo = AttnVec<T>::tr_read(base + v_rd[ot] + st * 16 * VPI);
      const vec4 hi = AttnVec<T>::tr_read(base + v_rd[ot] + (st * 16 + 8) * VPI);
      return join_halves<T>(lo, hi);
    };
    auto second_product = [&](lds_T* base) {
#pragma unroll
      for (int st = 0; st < 2 * KB; ++st)
#pragma unroll
        for (int ot = 0; ot < OT; ++ot) {
          const vec8 vf = read_v(base, st, ot);
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) oacc[qb][ot] = Tr::mfma32(vf, pf[qb][st], oacc[qb][ot]);
        }
    };

    for (int t = 0; t < n_tiles; ++t) {
      // K(t) and V(t - 1) have landed once only the younger loads are out; past the barrier everybody's have, and
      // nobody reads the stages of K(t - 1) and V(t - 2) any more
      attn_wait_vmcnt<(D - 1) * (Tile::KL / NWT + Tile::VL / NWT) + Tile::VL / NWT>();
      __builtin_amdgcn_s_barrier();
      issue(t + D);
      lds_T* const vb = (lds_T*)(sV + v_at * Tile::V_STAGE);
      const int nb = t * BNT + grp * BN;  // this group's first key
      if (nb < w_some) {
        f32x16 s[QB][KB];
        {
          lds_T* kb_ptr = (lds_T*)(sK + k_at * Tile::K_STAGE + k_rd);
          // (all reads first: left to itself the compiler fetches a pair and waits for it in front of every second product)
          vec8 kf[KB][KS];
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) kf[kb][ks] = *(lds_vec8*)(kb_ptr + kb * 32 * KPI + ks * 16);
          __builtin_amdgcn_sched_barrier(0x6);
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
              for (int qb = 0; qb < QB; ++qb) s[qb][kb] = Tr::mfma32(kf[kb][ks], qf[qb][ks], ks == 0 ? f32x16{} : s[qb][kb]);
            }
        }
        bool full = !ref_ok || nb + BN > w_every;
        if (!full) {
          float l_before[QB], mc[QB];
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) {
            l_before[qb] = l_run[qb];
            mc[qb] = -m_run[qb] * c;
          }
#pragma unroll
          for (int st = 0; st < 2 * KB; ++st) {
#pragma unroll
            for (int ot = 0; ot < OT; ++ot) {
              const vec8 vf = read_v(vb, st, ot);
#pragma unroll
              for (int qb = 0; qb < QB; ++qb) oacc[qb][ot] = Tr::mfma32(vf, pf[qb][st], oacc[qb][ot]);
            }
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
              for (int j = 0; j < 8; ++j)
                pf[qb][st][j] = Tr::from_float(
                    __builtin_amdgcn_exp2f(__builtin_fmaf(s[qb][st >> 1][(st & 1) * 8 + j], c, mc[qb])));
              l_run[qb] = add_elements(pf[qb][st], l_run[qb]);
            }
          }
          bool bad = false;
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) bad = bad || !(l_run[qb] <= kMaxRowSum);
          if (__builtin_expect(__builtin_amdgcn_ballot_w64(bad) != 0, 0)) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) l_run[qb] = l_before[qb];
            full = true;
            due = false;
          }
        }
        if (full) {
          if (due) second_product(vb);
          due = true;
          ref_ok = true;
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) {
            // lane holds keys nb + 32 kb + 8 g + 4 h + r (element 4 g + r of sub-block kb) of its query row
            const int q_row = w0 + qb * 32 + r32;
            const int left = (p.causal && q_row + 1 < N ? q_row + 1 : N) - nb - h * 4;
            float text = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
              for (int e = 0; e < 16; ++e) {
                float x = s[qb][kb][e];
                // a NaN score counts as -inf where the op says so (AttnParams::nan_reset)
                if (kb * 32 + (e >> 2) * 8 + (e & 3) >= left || (p.nan_reset != 0 && x != x)) x = -INFINITY;
                s[qb][kb][e] = x;
                text = fmaxf(text, x);
              }
            text = max_across_halves(text);
            // The reference point moves only when the row maximum has grown by more than kLazyLog2 binary orders since
            // it was last taken: until then P may exceed 1 by at most 2^kLazyLog2, harmless in fp32 sums and in P.
            constexpr float kLazyLog2 = 8.0f;
            const float m_cand = fmaxf(m_run[qb], text);
            const float drift = (m_run[qb] - m_cand) * c;  // <= 0; -inf (or NaN for inf - inf) on the first live tile
            const bool move = !(drift >= -kLazyLog2);
            const float m_new = move ? m_cand : m_run[qb];
            const float m_safe = __builtin_isinf(m_new) ? 0.0f : m_new;  // every key so far masked
            const float alpha = !move ? 1.0f : (__builtin_isinf(m_run[qb]) ? 0.0f : __builtin_amdgcn_exp2f(drift));
            const float mc = -m_safe * c;
            l_run[qb] *= alpha;
#pragma unroll
            for (int st = 0; st < 2 * KB; ++st) {
#pragma unroll
              for (int j = 0; j < 8; ++j)
                pf[qb][st][j] =
                    Tr::from_float(__builtin_amdgcn_exp2f(__builtin_fmaf(s[qb][st >> 1][(st & 1) * 8 + j], c, mc)));
              l_run[qb] = add_elements(pf[qb][st], l_run[qb]);
            }
            m_run[qb] = m_new;
            if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
              for (int ot = 0; ot < OT; ++ot)
#pragma unroll
                for (int e = 0; e < 16; ++e) oacc[qb][ot][e] *= alpha;
            }
            ref_ok = ref_ok && __builtin_amdgcn_ballot_w64(__builtin_isinf(m_new)) == 0;
          }
        }
      } else if (due) {
        second_product(vb);
        due = false;
      }
      k_at = k_at + 1 == NK ? 0 : k_at + 1;
      // (V(t): the stage behind V(t - 1)'s, which for t = 0 is none)
      if (t > 0) v_at = v_at + 1 == NV ? 0 : v_at + 1;
    }
    // the last tile's second product, when its V has landed; nothing is landing any more when the stages are reused
    attn_wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    if (due) second_product((lds_T*)(sV + v_at * Tile::V_STAGE));
    __syncthreads();

    // ---- wave groups: the other group hands its running state to group 0 through the ring's memory
    if constexpr (NG > 1) {
      static_assert(NG == 2, "the merge below pairs two groups");
      float* xch = reinterpret_cast<float*>(smem_raw) + wave * 64 + lane;
      constexpr int NVAL = 16 * OT + 2;
      if (grp == 1) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
          for (int ot = 0; ot < OT; ++ot)
#pragma unroll
            for (int e = 0; e < 16; ++e) xch[(qb * NVAL + ot * 16 + e) * NW * 64] = oacc[qb][ot][e];
          xch[(qb * NVAL + NVAL - 2) * NW * 64] = m_run[qb];
          xch[(qb * NVAL + NVAL - 1) * NW * 64] = l_run[qb];
        }
      }
      __syncthreads();
      if (grp == 0) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          const float m1 = xch[(qb * NVAL + NVAL - 2) * NW * 64];
          const float l1 = xch[(qb * NVAL + NVAL - 1) * NW * 64];
          // both states are sums of exp2((s - m) c) terms for their own reference m: bring them to the larger one
          const float m = fmaxf(m_run[qb], m1);
          const float a0 = __builtin_isinf(m_run[qb]) ? 0.0f : __builtin_amdgcn_exp2f((m_run[qb] - m) * c);
          const float a1 = __builtin_isinf(m1) ? 0.0f : __builtin_amdgcn_exp2f((m1 - m) * c);
          l_run[qb] = l_run[qb] * a0 + l1 * a1;
#pragma unroll
          for (int ot = 0; ot < OT; ++ot)
#pragma unroll
            for (int e = 0; e < 16; ++e)
              oacc[qb][ot][e] = oacc[qb][ot][e] * a0 + xch[(qb * NVAL + ot * 16 + e) * NW * 64] * a1;
        }
      }
      __syncthreads();
    }

    // ---- normalise and store permuted, out[b / G][m][b % G][o], through a strip of the wave's own: whole rows of
    // 16-byte pieces instead of 8 bytes of 64 rows at a time
    if (grp == 0) {
      T* const strip = reinterpret_cast<T*>(smem_raw) + wave * 32 * Tile::O_PITCH;
      // The arguments of the store are fetched here and not held over the loop, which has no registers for them: held, they and
      // by_heads had 18 scalar and 6 vector registers spilled at head dim 64 with four workgroups per CU (3 and 5 where by_heads
      // was no argument), 4 and none so.  us, held -> fetched: 64 x 12 x 384^2, d 64, mixed lengths 32.3 -> 29.6, 64 x 12 x 512^2
      // 73.2 -> 69.9, 4 x 8 x 2048^2, d 80 57.1 -> 55.4.  Held are M and O with four workgroups per CU (fetched: 9 vector registers)
      // and all at head dims to 128 (2 x 16 x 4096^2 277.2, fetched 278.6).
      const AttnParams& w = KS == 8 ? p : arguments_anew<AttnParams>();
      const AttnParams& extent = Tile::OCC >= 4 ? p : w;
      const int out_seq = quotient(b, w.by_heads);
      T* const ob = reinterpret_cast<T*>(w.out) + ((int64_t)out_seq * w.M * w.G + (b - out_seq * w.G)) * w.O;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const int q_row = w0 + qb * 32 + r32;
        const float l_tot = sum_across_halves(l_run[qb]);
        const float inv = (l_tot > 0.0f && q_row < m_rows) ? 1.0f / l_tot : 0.0f;
#pragma unroll
        for (int ot = 0; ot < OT; ++ot)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            vec4 ov;
#pragma unroll
            for (int j = 0; j < 4; ++j) ov[j] = Tr::from_float(oacc[qb][ot][g * 4 + j] * inv);
            *reinterpret_cast<vec4*>(strip + r32 * Tile::O_PITCH + ot * 32 + g * 8 + h * 4) = ov;
          }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        constexpr int OC = Tile::OP / 8;
#pragma unroll
        for (int i = 0; i < OC / 2; ++i) {
          const int idx = i * 64 + lane, row = idx / OC, ch = idx - row * OC;
          const int m = w0 + qb * 32 + row;
          if (m < extent.M && ch * 8 < extent.O)
            store_vec(ob + (int64_t)m * w.G * w.O + ch * 8, *reinterpret_cast<const vec8*>(strip + row * Tile::O_PITCH + ch * 8));
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    }
    if (passes > 1 || p.entries < p.B) __syncthreads();  // the strips lie where the next tiles land
  }
}

}  // namespace aitamd
