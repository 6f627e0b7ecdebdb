// Stage 2's selection test as a threshold on the raw dot product of pooled query and key.
//
// The test "float(round16(raw * scale)) + theta >= anchor" is monotone in raw, so for every pooled row there is one float32 x* with
// "test passes  <=>  raw >= x*".  x* is found by search over the ordered float32 bit patterns, evaluating the test exactly as
// written.  All lanes of a row test as many points at a time: one lane to a row (bisection, 32 dependent
// rounds) was a launch of 4.8 us at any size, 64 lanes need six rounds and fit beside the pooling in stage 1's epilogue.
#pragma once
#include "aa_common.h"

namespace aa {

__device__ __forceinline__ float ordered_to_float(const uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);  // monotone bijection uint32 -> float32
}

// The lanes for which the test passes for x; round16 rounds to the tensors' 16-bit type, non-strict float32 compare.  (The compare is written out:
// it is false for NaN also where the compiler is told that there is none.)
template <typename T>
__device__ __forceinline__ uint64_t select_test(const float x, const float scale2, const float theta, const float anchor) {
  const float sum = T::round_product(x, scale2) + theta;  // the score as (dot * scale).to(dtype) evaluates it for this type
  uint64_t lanes;
  asm volatile("v_cmp_ge_f32_e64 %0, %1, %2" : "=s"(lanes) : "v"(sum), "v"(anchor));
  return lanes;
}

// Smallest float32 x that passes, as bits (NaN if there is none, which compares false with everything).  `lanes` (a power of
// two, at most 64) neighbouring lanes share a row; all lanes of the wave must be active and take part.
template <typename T>
__device__ __forceinline__ uint32_t select_threshold(const float anchor, const float scale2, const float theta, const int lane, const int lanes) {
  // ordered keys: 0x007fffff <-> -inf, 0xff800000 <-> +inf (NaNs lie outside that range)
  uint32_t lo = 0x007fffffu, hi = 0xff800000u;
  const uint32_t j = (uint32_t)(lane & (lanes - 1));
  const int first = lane - (int)j, bits = __ffs(lanes) - 1;
  const uint64_t own = lanes == 64 ? ~0ull : (1ull << lanes) - 1ull;
  const bool exists = (select_test<T>(ordered_to_float(hi), scale2, theta, anchor) >> lane) & 1ull;
  while (__any(lo < hi)) {  // invariant, if there is a solution: hi passes, what lies below lo does not
    const uint32_t step = ((hi - lo) >> bits) + 1u;
    const uint64_t pass = (select_test<T>(ordered_to_float(min(lo + j * step, hi)), scale2, theta, anchor) >> first) & own;
    const uint32_t f = pass != 0ull ? (uint32_t)__ffsll((unsigned long long)pass) - 1u : (uint32_t)lanes;  // the first point that passes
    const uint32_t above = f > 0u ? min(lo + (f - 1u) * step, hi) + 1u : lo;
    if (pass != 0ull) hi = min(lo + f * step, hi);
    lo = above;
  }
  return exists ? __float_as_uint(ordered_to_float(hi)) : 0x7fc00000u;
}

}  // namespace aa
