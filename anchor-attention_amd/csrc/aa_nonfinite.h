// P.V where V is not finite, for the kernels that keep a probability as two 16-bit numbers (rows, masked and decode).
//
// With one product per key an infinite V gives an infinity.  With two it gives NaN: the rest of a probability may be 0 or
// negative, and so are the keys past the last one, which repeat its row.  A wave that finds NaN among its sums therefore forms them once
// more here: the rest meets V with its infinities and NaN left out, keys past the end count as 0 and a positive probability
// does not round to 0.  What is NaN after that is NaN in float32 as well: a V that is, infinities of both signs, and an infinity at
// a key of probability 0 (a masked key whose tile other rows of the work-group see).
//
// The operands come straight from memory, V two bytes at a time: some tens of times slower than the kernels' own tiles, and
// reached by such V only.  The others pay one addition per accumulator register: 777 rows over 777 keys 22.40 -> 22.49 us, a
// decode step over 33001 keys 32.25 -> 32.53, a padded batch of 3 x 2500 189.2 -> 189.7 (32/8 heads of 128).
#pragma once
#include "aa_common.h"

namespace aa {

__device__ __forceinline__ bool is_nan(float x) {
  asm volatile("" : "+v"(x));  // (also where the compiler is told that there is none)
  return (__float_as_uint(x) & 0x7fffffffu) > 0x7f800000u;
}

// whether an accumulator of this lane is NaN (infinities of both signs count too)
template <int N>
__device__ __forceinline__ bool holds_nan(const floatx16 (&acc)[N]) {
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int db = 0; db < N; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[r & 3] += acc[db][r];
  return is_nan((sum[0] + sum[1]) + (sum[2] + sum[3]));
}

// Adds the 32 keys from key0 on to acc (O^T, layout of the kernels).  `seen`: bit j says whether this lane's column sees
// key0 + j (no bit of a key from n_keys on is set); m_base: the column's final maximum; qreg: its query.
template <typename T, int D>
__device__ __forceinline__ void exact_pv_tile(floatx16 (&acc)[D / 32], const typename T::vec8 (&qreg)[D / 16], const char* kbase, const char* vbase,
                                              const uint32_t k_row_bytes, const uint32_t v_row_bytes, const int key0, const int n_keys,
                                              const uint32_t seen, const float m_base, const float scale, const int lane) {
  typedef typename T::vec8 vec8;
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
  const int half = lane >> 5, c32 = lane & 31;
  const char* kp = kbase + (uint64_t)(uint32_t)min(key0 + c32, n_keys - 1) * k_row_bytes + 16 * half;
  floatx16 s;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) s = T::mfma(*reinterpret_cast<const vec8*>(kp + 32 * ks), qreg[ks], s);
  u32x4 pw[2], pw_rest[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) {  // accumulator registers 2i, 2i+1
    const int j = 8 * (i >> 1) + 4 * half + 2 * (i & 1);
    const float e0 = (seen >> j) & 1u ? prob_exp2<T>(s[2 * i] - m_base, scale) : 0.f;
    const float e1 = (seen >> (j + 1)) & 1u ? prob_exp2<T>(s[2 * i + 1] - m_base, scale) : 0.f;
    uint32_t w = T::pack(e0, e1);
    if (e0 > 0.f && (w & 0xffffu) == 0u) w |= 1u;
    if (e1 > 0.f && (w >> 16) == 0u) w |= 0x10000u;
    pw[i >> 2][i & 3] = w;
    pw_rest[i >> 2][i & 3] = T::pack_rest(e0, e1, w);
  }
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      u16x8 v, finite;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int key = key0 + 16 * st + 8 * (e >> 2) + 4 * half + (e & 3);
        const uint16_t x = *reinterpret_cast<const uint16_t*>(vbase + (uint64_t)(uint32_t)min(key, n_keys - 1) * v_row_bytes + 2 * (32 * db + c32));
        v[e] = key < n_keys ? x : (uint16_t)0;
        finite[e] = (v[e] & T::kExponent) == T::kExponent ? (uint16_t)0 : v[e];
      }
      acc[db] = T::mfma(*reinterpret_cast<const vec8*>(&v), *reinterpret_cast<const vec8*>(&pw[st]), acc[db]);
      acc[db] = T::mfma(*reinterpret_cast<const vec8*>(&finite), *reinterpret_cast<const vec8*>(&pw_rest[st]), acc[db]);
    }
}

}  // namespace aa
