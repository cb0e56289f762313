// Packed 16-bit helpers of the two-tasks-per-lane kernels: one task in each
// half of a register.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

namespace bsx {

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
typedef const uint32_t __attribute__((address_space(1))) * gdword;

__device__ __forceinline__ u16x2 pk(uint32_t x) { return __builtin_bit_cast(u16x2, x); }
__device__ __forceinline__ uint32_t pku(u16x2 x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ i16x2 pks(u16x2 x) { return __builtin_bit_cast(i16x2, x); }
__device__ __forceinline__ u16x2 pkmax(u16x2 a, u16x2 b) { return __builtin_elementwise_max(a, b); }
__device__ __forceinline__ u16x2 pkmin(u16x2 a, u16x2 b) { return __builtin_elementwise_min(a, b); }
__device__ __forceinline__ u16x2 pksat(u16x2 a, u16x2 b) { return __builtin_elementwise_sub_sat(a, b); }
__device__ __forceinline__ u16x2 pk2(int lo, int hi) { return pk((uint32_t)(lo & 0xffff) | (uint32_t)hi << 16); }
__device__ __forceinline__ u16x2 splat(uint32_t x) { return pk(x | x << 16); }
// 0xffff in every half whose signed value is negative
__device__ __forceinline__ uint32_t negmask(u16x2 x) { return __builtin_bit_cast(uint32_t, pks(x) >> (int16_t)15); }
__device__ __forceinline__ u16x2 sel(uint32_t m, u16x2 a, u16x2 b) { return pk((pku(a) & m) | (pku(b) & ~m)); }
// signed forms
__device__ __forceinline__ u16x2 smax(u16x2 a, u16x2 b) {
  return __builtin_bit_cast(u16x2, __builtin_elementwise_max(pks(a), pks(b)));
}
__device__ __forceinline__ u16x2 smin(u16x2 a, u16x2 b) {
  return __builtin_bit_cast(u16x2, __builtin_elementwise_min(pks(a), pks(b)));
}
__device__ __forceinline__ u16x2 ssat(u16x2 a, u16x2 b) {
  return __builtin_bit_cast(u16x2, __builtin_elementwise_sub_sat(pks(a), pks(b)));
}

// A uniform constant in both halves whose value the compiler does not see: it
// would turn min(x, 1) into a compare and a select per half, a multiply by a
// power of two into shifts, and a chain of subtractions into one constant each.
__device__ __forceinline__ u16x2 hidden(uint32_t x) {
  uint32_t v = x | x << 16;
  asm("" : "+s"(v));
  return pk(v);
}

// f(0), f(1), ... with compile-time arguments (a long loop is not unrolled)
template <class F, int... I>
__device__ __forceinline__ void for_each_index(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// A byte sequence read as aligned dwords; indices are clamped to the dwords
// that hold its bytes.
struct DwordSeq {
  gdword p;
  int sh, last;
  __device__ __forceinline__ void set(const uint8_t* base, int len) {
    const uintptr_t a = (uintptr_t)base;
    p = (gdword)(a & ~(uintptr_t)3);
    sh = (int)(a & 3);
    last = (sh + (len > 0 ? len : 1) - 1) >> 2;
  }
  __device__ __forceinline__ uint32_t at(int d) const { return p[d < 0 ? 0 : d < last ? d : last]; }
};

}  // namespace bsx
