// C ABI launcher of the fused attention kernel (bmm_softmax_bmm_permute).
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "../../include/aitemplate_amd_kernels.h"
#include "attention_form.hpp"
#include "attention_kernel.hpp"
#include "attention_pipe.hpp"
#include "device.hpp"
#include "errors.hpp"

namespace aitamd {
namespace {

constexpr int kMaxDevices = 64;

// Variant forced by aitamd_attention_set_variant: -1 automatic, 0..4 a Form (attention_form.hpp).  The environment variable
// AITAMD_ATTN_MODE gives the initial value and is read once, not on every launch.
constexpr int kVariantUnset = -2;
std::atomic<int> g_forced_variant{kVariantUnset};
int forced_variant() {
  int m = g_forced_variant.load(std::memory_order_relaxed);
  if (m == kVariantUnset) {
    const char* env = getenv("AITAMD_ATTN_MODE");
    const int from_env = env ? atoi(env) : -1;
    g_forced_variant.compare_exchange_strong(m, from_env >= 0 && from_env <= kRows64 ? from_env : -1);
    m = g_forced_variant.load(std::memory_order_relaxed);
  }
  return m;
}

template <int KS, int OT, int FORM>
struct PipeOf {
  static constexpr bool kNarrow = KS <= 4 && OT <= 2;
  using type = std::conditional_t<
      FORM == kRows256 && kNarrow, AttnPipe<KS, OT, 1, 4, kNarrow ? 2 : 1, 1, 1, 2>,
      std::conditional_t<FORM == kGroups, AttnPipe<KS, OT, kNarrow ? 2 : 1, 4, 1, 2, 1, 2>,
                         std::conditional_t<FORM == kSmall, AttnPipe<KS, OT, 1, 2, 1, 2, 1, 2>,
                                            std::conditional_t<FORM == kRows64, AttnPipe<KS, OT, 1, 2, 1, 1, 1, 2>,
                                                               AttnPipe<KS, OT, 1, 4, 1, 1, 1, kNarrow ? 4 : 2>>>>>;
};

// the kernel's opt-in to more than 64 KiB of LDS, once per device; the outcome is kept: a failed opt-in must fail every
// later call too, not only the first
struct LdsOptIn {
  std::once_flag once[kMaxDevices];
  hipError_t err[kMaxDevices];
  hipError_t operator()(const void* kernel, int bytes) {
    int dev = 0;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    dev %= kMaxDevices;
    std::call_once(once[dev], [&] { err[dev] = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes); });
    return err[dev];
  }
};

template <class T, int KS, int OT, int FORM>
hipError_t launch_pipe(const AttnParams& p_in, hipStream_t stream) {
  using Tile = typename PipeOf<KS, OT, FORM>::type;
  auto kernel = attention_pipe_kernel<T, Tile>;
  static LdsOptIn opt_in;
  const hipError_t e = opt_in(reinterpret_cast<const void*>(kernel), Tile::kLdsBytes);
  if (e != hipSuccess) return e;
  AttnParams p = p_in;
  int64_t m_tiles = ((int64_t)p.M + Tile::BM - 1) / Tile::BM;
  if (p.paired) m_tiles = (m_tiles + 1) / 2;
  p.tiles = (int32_t)m_tiles;
  p.entries = p.B < 65535 ? p.B : 65535;
  p.dealt = p.entries == p.B && m_tiles * p.B <= 0x7fffffffll;
  p.by_tiles = make_divisor(m_tiles);
  p.by_heads = make_divisor(p.G);
  dim3 grid((unsigned)p.tiles, (unsigned)p.entries, 1);
  hipLaunchKernelGGL(kernel, grid, dim3(Tile::NT), Tile::kLdsBytes, stream, p);
  return hipGetLastError();
}

// operands that do not come in whole, aligned 16-byte pieces (VEC: that do, in matrices beyond 32-bit offsets)
template <class T, int KS, int OT, bool VEC>
hipError_t launch_staged(const AttnParams& p, hipStream_t stream) {
  using Tile = AttnTile<KS, OT>;
  auto kernel = attention_kernel<T, Tile, VEC>;
  static LdsOptIn opt_in;
  const hipError_t e = opt_in(reinterpret_cast<const void*>(kernel), Tile::kLdsBytes);
  if (e != hipSuccess) return e;
  const int64_t m_tiles = (p.M + Tile::BM - 1) / Tile::BM;
  dim3 grid((unsigned)m_tiles, (unsigned)(p.B < 65535 ? p.B : 65535), 1);
  hipLaunchKernelGGL(kernel, grid, dim3(Tile::NT), Tile::kLdsBytes, stream, p);
  return hipGetLastError();
}

typedef hipError_t (*AttnLaunch)(const AttnParams&, hipStream_t);

// smallest padded head dims first; (K <= 16 KS, O <= 32 OT); 160: the deepest attention of Stable Diffusion v1 (1280
// channels, 8 heads)
#define AITAMD_ATTN_DIMS(X) X(2, 1) X(3, 2) X(4, 2) X(4, 4) X(6, 3) X(8, 4) X(10, 5)
template <class T, int FORM>
AttnLaunch pick_pipe(int ks, int ot) {
#define AITAMD_ATTN_CASE(KS, OT) \
  if (ks <= KS && ot <= OT) return &launch_pipe<T, KS, OT, FORM>;
  AITAMD_ATTN_DIMS(AITAMD_ATTN_CASE)
#undef AITAMD_ATTN_CASE
  return nullptr;
}
template <class T>
AttnLaunch pick_pipe(int form, int ks, int ot) {
  switch (form) {
    case kRows256: return pick_pipe<T, kRows256>(ks, ot);
    case kGroups: return pick_pipe<T, kGroups>(ks, ot);
    case kSmall: return pick_pipe<T, kSmall>(ks, ot);
    case kRows64: return pick_pipe<T, kRows64>(ks, ot);
    default: return pick_pipe<T, kRows128>(ks, ot);
  }
}
template <class T, bool VEC>
AttnLaunch pick_staged(int ks, int ot) {
#define AITAMD_ATTN_CASE(KS, OT) \
  if (ks <= KS && ot <= OT) return &launch_staged<T, KS, OT, VEC>;
  AITAMD_ATTN_DIMS(AITAMD_ATTN_CASE)
#undef AITAMD_ATTN_CASE
  return nullptr;
}

// x rounded to the nearest fp16 (dtype 0) or bf16 value, ties to even, as a float.  Done on the bits: host-side
// conversions through _Float16 / __bf16 would call compiler-runtime routines that a model library linked by the
// host C++ compiler does not have.
float round_to_elem(float x, int dtype) {
  uint32_t u;
  memcpy(&u, &x, 4);
  const uint32_t sign = u & 0x80000000u, mag = u & 0x7fffffffu;
  if (mag >= 0x7f800000u) return x;  // infinities and NaNs stay what they are
  uint32_t r;
  if (dtype != 0) {
    r = mag + 0x7fffu + ((mag >> 16) & 1u);  // keep 8 bits of mantissa
    r &= 0xffff0000u;
  } else {
    const int e = (int)(mag >> 23) - 127;
    if (e > 15) {
      r = 0x7f800000u;  // beyond the largest half
    } else if (e >= -14) {
      r = mag + 0xfffu + ((mag >> 13) & 1u);  // normal half: keep 10 bits of mantissa
      r &= 0xffffe000u;
      if (r >= 0x47800000u) r = 0x7f800000u;  // rounded up past 65504
    } else {
      // subnormal half: a multiple of 2^-24
      float f;
      memcpy(&f, &mag, 4);
      const float q = f * 16777216.0f;          // exact scaling
      const float n = __builtin_rintf(q);       // ties to even in the default rounding mode
      f = n * (1.0f / 16777216.0f);
      memcpy(&r, &f, 4);
    }
  }
  r |= sign;
  float out;
  memcpy(&out, &r, 4);
  return out;
}

}  // namespace
}  // namespace aitamd

using namespace aitamd;

namespace {

int attention_entry(const char* who, int dtype, const void* q, const void* k, const void* v, void* out, int64_t B,
                    int64_t M, int64_t N, int64_t K, int64_t O, int64_t G, float scale, int causal,
                    const int32_t* kv_len, const int32_t* q_len, bool nan_reset, void* stream) {
  if (dtype != 0 && dtype != 1) return fail("%s: bad dtype %d", who, dtype);
  if (B < 0 || M < 0 || N < 0 || K < 0 || O < 0) return fail("%s: negative dimension", who);
  if (G <= 0 || (B % G) != 0) return fail("%s: batch %lld is not a multiple of heads %lld", who,
                                          (long long)B, (long long)G);
  if (B == 0 || M == 0 || O == 0) return 0;
  if (B > 0x7fffffffll || M > 0x7fffffffll || N > 0x7fffffffll) return fail("%s: dimension too large", who);
  if (K > 160 || O > 160) return fail("%s: head dims above 160 are not supported (K=%lld O=%lld)", who,
                                      (long long)K, (long long)O);
  if (!out || (N > 0 && (!q || !k || !v))) return fail("%s: null pointer", who);
  AttnParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = out;
  p.B = (int32_t)B;
  p.M = (int32_t)M;
  p.N = (int32_t)N;
  p.K = N > 0 ? (int32_t)K : 0;  // (no keys: q, which may be null then, is not read)
  p.O = (int32_t)O;
  p.G = (int32_t)G;
  // the reference hands alpha to its kernel in the element type
  // (python/aitemplate/backend/rocm/gemm/bmm_softmax_bmm_permute.py:47-51)
  p.scale_log2e = round_to_elem(scale, dtype) * 1.4426950408889634f;
  p.causal = causal ? 1 : 0;
  p.kv_len = kv_len;
  p.q_len = q_len;
  p.nan_reset = nan_reset ? 1 : 0;
  const int ks = (int)((K + 15) / 16) > 0 ? (int)((K + 15) / 16) : 1;
  const int ot = (int)((O + 31) / 32);
  const bool vec = (K % 8 == 0) && (O % 8 == 0) && ((reinterpret_cast<uintptr_t>(q) & 15) == 0) &&
      ((reinterpret_cast<uintptr_t>(k) & 15) == 0) && ((reinterpret_cast<uintptr_t>(v) & 15) == 0);
  // direct-to-LDS tiles address K and V of one batch entry with 32-bit byte offsets
  const int64_t kv_dim = K > O ? K : O;
  // (tiles are issued past the last one, and out-of-range offsets are the largest of these and 2^31 added up)
  const bool dma = vec && (N + 4 * 128) * kv_dim * 2 < 0x70000000;
  AttnLaunch fn = nullptr;
  if (dma) {
    int form = choose_form(B, M, N, ks, ot, causal != 0, current_device_cus(), &p.paired);
    // aitamd_attention_set_variant(0|1|2|3|4) forces a form (a test and measurement knob)
    if (forced_variant() >= 0) form = forced_variant();
    if (form == kRows256) p.paired = 0;
    fn = dtype == 0 ? pick_pipe<f16>(form, ks, ot) : pick_pipe<bf16>(form, ks, ot);
  } else if (dtype == 0) {
    fn = vec ? pick_staged<f16, true>(ks, ot) : pick_staged<f16, false>(ks, ot);
  } else {
    fn = vec ? pick_staged<bf16, true>(ks, ot) : pick_staged<bf16, false>(ks, ot);
  }
  if (!fn) return fail("%s: no instance for K=%lld O=%lld", who, (long long)K, (long long)O);
  const hipError_t e = fn(p, reinterpret_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail("%s: launch failed: %s", who, hipGetErrorString(e));
  return 0;
}

}  // namespace

extern "C" int aitamd_attention_set_variant(int variant) {
  if (variant < -1 || variant > kRows64)
    return fail("aitamd_attention_set_variant: variant %d is not one of -1, 0, 1, 2, 3, 4", variant);
  g_forced_variant.store(variant, std::memory_order_relaxed);
  return 0;
}

extern "C" int aitamd_bmm_softmax_bmm_permute(int dtype, const void* q, const void* k, const void* v, void* out,
                                              int64_t B, int64_t M, int64_t N, int64_t K, int64_t O, int64_t G,
                                              float scale, int causal, void* stream) {
  // NaN scores count as -inf: the reference gives this op's kernel ScaleAndResetNaNToMinusInfinity
  // (python/aitemplate/backend/rocm/gemm/bmm_softmax_bmm_permute.py:106, bmm_softmax_bmm.py:99)
  return attention_entry("aitamd_bmm_softmax_bmm_permute", dtype, q, k, v, out, B, M, N, K, O, G, scale, causal, nullptr,
                         nullptr, true, stream);
}

extern "C" int aitamd_mem_eff_attention(int dtype, const void* q, const void* k, const void* v, void* out,
                                        int64_t batch, int64_t heads, int64_t seq_q, int64_t seq_kv, int64_t head_dim,
                                        int64_t head_dim_v, float scale, int causal, const int32_t* lengths_kv,
                                        const int32_t* lengths_q, void* stream) {
  if (batch < 0 || heads <= 0) return fail("aitamd_mem_eff_attention: bad batch %lld or heads %lld", (long long)batch,
                                           (long long)heads);
  if (batch > 0x7fffffffll / heads) return fail("aitamd_mem_eff_attention: dimension too large");
  // (a NaN score stays a NaN: the reference's kernel for this op scales only,
  // python/aitemplate/backend/rocm/attention/mem_eff_attention.py:74)
  return attention_entry("aitamd_mem_eff_attention", dtype, q, k, v, out, batch * heads, seq_q, seq_kv, head_dim,
                         head_dim_v, heads, scale, causal, lengths_kv, lengths_q, false, stream);
}
