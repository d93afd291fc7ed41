// Shared device-side vocabulary for the gfx950 GEMM-family kernels: vector
// types, buffer-resource helpers, fp16/bf16 conversion and the XCD-aware
// workgroup -> output-tile mapping.  gfx950 (MI355X, CDNA4) only.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace aitamd {

using f16 = _Float16;
using bf16 = __bf16;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

#define AITAMD_DEVICE __device__ __forceinline__

constexpr int kWaveSize = 64;
constexpr int kNumXcd = 8;  // MI355X: 8 accelerator dies, one L2 each

// ---------------------------------------------------------------------------
// Element-type traits: 8-wide operand vector and the 32x32x16 / 16x16x32 MFMA.
// ---------------------------------------------------------------------------
template <class T>
struct ElemTraits;

template <>
struct ElemTraits<f16> {
  using vec8 = f16x8;
  using vec4 = f16x4;
  static AITAMD_DEVICE f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static AITAMD_DEVICE f32x4 mfma16(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static AITAMD_DEVICE float to_float(f16 v) { return (float)v; }
  static AITAMD_DEVICE f16 from_float(float v) { return (f16)v; }
  // float(v) + c in one instruction: with `one` = 1.0 in a register the compiler cannot see through, the fused
  // multiply-add of a widened half maps to v_fma_mix_f32 (conversion and add together; same single rounding)
  static AITAMD_DEVICE float to_float_plus(f16 v, float one, float c) { return __builtin_fmaf((float)v, one, c); }
};

template <>
struct ElemTraits<bf16> {
  using vec8 = bf16x8;
  using vec4 = bf16x4;
  static AITAMD_DEVICE f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static AITAMD_DEVICE f32x4 mfma16(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static AITAMD_DEVICE float to_float(bf16 v) { return (float)v; }
  static AITAMD_DEVICE bf16 from_float(float v) { return (bf16)v; }
  static AITAMD_DEVICE float to_float_plus(bf16 v, float one, float c) { (void)one; return (float)v + c; }
};

// LDS transpose read: 4 x 16-bit per lane, gathered across the 16 lanes of a block.
// __restrict__ is for the compiler's wait insertion: without alias information on the read it assumes that any
// direct-to-LDS load on its way may be the data and drains them all (s_waitcnt vmcnt(0)) in front of every read, which
// took the prefetch distance of every kernel that uses this away (bmm crr 16 x 208 x 24, K = 832: 102 us, 55 without).
AITAMD_DEVICE f16x4 tr_read16(const f16* __restrict__ p) {
  typedef __fp16 raw4 __attribute__((__vector_size__(4 * sizeof(__fp16))));
  const raw4 r = __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) raw4*)p);
  return __builtin_bit_cast(f16x4, r);
}
AITAMD_DEVICE bf16x4 tr_read16(const bf16* __restrict__ p) {
  typedef __bf16 raw4 __attribute__((__vector_size__(4 * sizeof(__bf16))));
  const raw4 r = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) raw4*)p);
  return __builtin_bit_cast(bf16x4, r);
}
template <class T>
AITAMD_DEVICE typename ElemTraits<T>::vec8 join_halves(typename ElemTraits<T>::vec4 lo, typename ElemTraits<T>::vec4 hi) {
  typename ElemTraits<T>::vec8 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[j] = lo[j];
    v[4 + j] = hi[j];
  }
  return v;
}

// ---------------------------------------------------------------------------
// Raw buffer resources.  Loads whose byte offset is >= num_records return 0,
// which is how every M/N/K tail is zero-filled without branches.
// ---------------------------------------------------------------------------
// f(integral_constant<int, I>) for I in [I0, I1): a loop whose index is a constant expression in the body
// (immediate operands of builtins)
template <int I0, int I1, class F>
AITAMD_DEVICE void static_for(F&& f) {
  if constexpr (I0 < I1) {
    f(std::integral_constant<int, I0>{});
    static_for<I0 + 1, I1>(f);
  }
}

constexpr uint32_t kOobOffset = 0x80000000u;  // >= any num_records we build

// Every descriptor in these kernels is the same for all lanes of a wave (one per tile, batch entry or wave
// part), but the compiler cannot prove that for values computed from the wave index or loaded tile coordinates,
// and a buffer access through a descriptor it takes for lane-varying is wrapped in a loop over the wave's
// distinct descriptors (four v_readfirstlane, two 64-bit compares and a branch per access).  Reading base and
// size from the first lane states the uniformity; where they already are scalar registers this folds away.
AITAMD_DEVICE __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t num_bytes) {
  const uint64_t v = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), 0,
                                           __builtin_amdgcn_readfirstlane(num_bytes), 0x00020000);
}

AITAMD_DEVICE u32x4 buffer_load_16B(__amdgpu_buffer_rsrc_t r, uint32_t voffset) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, voffset, 0, 0);
}
AITAMD_DEVICE uint32_t buffer_load_4B(__amdgpu_buffer_rsrc_t r, uint32_t voffset) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, voffset, 0, 0);
}

// A vector at an address of element alignment: one load or store (the gfx950 target reads and writes global memory
// at any alignment)
template <class V, class T>
AITAMD_DEVICE V load_vec(const T* p) {
  V v;
  __builtin_memcpy(&v, p, sizeof(V));
  return v;
}
template <class V, class T>
AITAMD_DEVICE void store_vec(T* p, V v) {
  __builtin_memcpy(p, &v, sizeof(V));
}

// Clamp a 64-bit byte count into the 32-bit num_records field.
AITAMD_DEVICE uint32_t clamp_records(int64_t bytes) {
  return bytes <= 0 ? 0u : (bytes >= 0x7fffffffll ? 0x7fffffffu : (uint32_t)bytes);
}

// ---------------------------------------------------------------------------
// Division by a number the host knows: the quotient by a multiplication with its scaled reciprocal (Granlund and
// Montgomery, "Division by invariant integers using multiplication", 1994), three scalar instructions.  The compiler's own
// division of two values in registers is a chain of 35, through the vector unit and back, and a tile's coordinates took
// three of them ahead of its first load.
// ---------------------------------------------------------------------------
struct Divisor {
  uint32_t mul, shift;
};
// d of 1 to 2^31 - 1
constexpr Divisor make_divisor(int64_t d) {
  uint32_t shift = 0;
  while ((1ll << shift) < d) ++shift;
  return {(uint32_t)((((1ull << shift) - (uint64_t)d) << 32) / (uint64_t)d + 1), shift};
}
// n / d for n of 0 to 2^31 - 1 (mulhi(n, mul) <= n: the sum stays below 2^32)
constexpr __host__ __device__ __forceinline__ int quotient(int n, Divisor d) {
  const uint32_t hi = (uint32_t)(((uint64_t)(uint32_t)n * d.mul) >> 32);
  return (int)((hi + (uint32_t)n) >> d.shift);
}
constexpr bool divides_right(long long d) {
  const Divisor r = make_divisor(d);
  for (long long q : {0ll, 1ll, 2ll, 3ll, 0x7fffffffll / d - 1, 0x7fffffffll / d})
    for (long long n : {q * d - 1, q * d, q * d + 1, q * d + d - 1})
      if (n >= 0 && n <= 0x7fffffffll && quotient((int)n, r) != n / d) return false;
  return quotient(0x7fffffff, r) == 0x7fffffffll / d;
}
static_assert(divides_right(1) && divides_right(2) && divides_right(3) && divides_right(7) && divides_right(8) && divides_right(641) &&
              divides_right(65535) && divides_right(65536) && divides_right(65537) && divides_right(0x3fffffff) &&
              divides_right(0x40000000) && divides_right(0x40000001) && divides_right(0x7ffffffe) && divides_right(0x7fffffff));

// The arguments of a kernel whose one parameter is a P, as memory that nothing is known of: what is read through this is
// fetched where it is used.  The compiler fetches an argument at the kernel's start and holds it in registers to its last
// use; where that is behind a long loop, it stands in the loop's way, and what does not fit is spilled.
template <class P>
AITAMD_DEVICE const P& arguments_anew() {
  typedef const __attribute__((address_space(4))) P* scalar_ptr;
  uintptr_t at = (uintptr_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(at));
  return *(const P*)(scalar_ptr)at;
}

}  // namespace aitamd
