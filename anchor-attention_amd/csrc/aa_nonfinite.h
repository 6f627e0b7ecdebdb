// P.V where its sums are not finite, for the kernels that keep a probability as two 16-bit numbers (rows, masked and decode).
//
// With one product per key an infinite V gives an infinity.  With two it gives NaN: the rest of a probability may be 0 or
// negative, and so are the keys past the last one, which repeat its row.  A wave that finds NaN among its sums therefore forms them once
// more here: the rest meets V with its infinities and NaN left out, keys past the end count as 0 and a positive probability
// does not round to 0.  What is NaN after that is NaN in float32 as well: a V that is, infinities of both signs, and an infinity at
// a key of probability 0 (a masked key whose tile other rows of the work-group see).
//
// The bf16 rows and masked modes' probabilities are relative to a score that may lie up to 14 bits below the row's max (aa_flash.hip): 32 keys
// sum to as much as 2^15, and P.V overflows float32 from |V| = 3.4e38 / (1024 n) on for n keys.  There a wave that finds infinities
// among its sums comes here too and takes the row's max first, so that V may be as large as with probabilities up to 1, 3.4e38 / n.
//
// The operands come straight from memory, V two bytes at a time: some tens of times slower than the kernels' own tiles, and
// reached by such V only.  The others pay one addition per accumulator register: 777 rows over 777 keys 22.40 -> 22.49 us, a
// decode step over 33001 keys 32.25 -> 32.53, a padded batch of 3 x 2500 189.2 -> 189.7 (32/8 heads of 128).
#pragma once
#include "aa_common.h"

namespace aa {

// The bits of a float without its sign, hidden from the compiler: where it is told that there is no NaN, it would make of a comparison
// of them one of floats, which NaN does not pass.
__device__ __forceinline__ uint32_t magnitude_bits(const float x) {
  uint32_t bits = __float_as_uint(x) & 0x7fffffffu;
  asm volatile("" : "+v"(bits));
  return bits;
}
__device__ __forceinline__ bool is_nan(const float x) { return magnitude_bits(x) > 0x7f800000u; }
__device__ __forceinline__ bool is_finite(const float x) { return magnitude_bits(x) < 0x7f800000u; }

// NaN if an accumulator of this lane is NaN or infinities of both signs are among them, infinite or NaN if one of them is infinite
template <int N>
__device__ __forceinline__ float sum_of_all(const floatx16 (&acc)[N]) {
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int db = 0; db < N; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[r & 3] += acc[db][r];
  return (sum[0] + sum[1]) + (sum[2] + sum[3]);
}

// Raw scores of the 32 keys from key0 on (S^T, layout of the kernels).
template <typename T, int D>
__device__ __forceinline__ floatx16 exact_scores(const typename T::vec8 (&qreg)[D / 16], const char* kbase, const uint32_t k_row_bytes, const int key0,
                                                 const int n_keys, const int lane) {
  const char* kp = kbase + (uint64_t)(uint32_t)min(key0 + (lane & 31), n_keys - 1) * k_row_bytes + 16 * (lane >> 5);
  floatx16 s;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) s = T::mfma(*reinterpret_cast<const typename T::vec8*>(kp + 32 * ks), qreg[ks], s);
  return s;
}

// The largest of them that this lane holds and its column sees (`seen`: as below), or `mx`.
__device__ __forceinline__ float exact_max(const floatx16& s, const uint32_t seen, const int lane, float mx) {
#pragma unroll
  for (int r = 0; r < 16; ++r)
    if ((seen >> (8 * (r >> 2) + 4 * (lane >> 5) + (r & 3))) & 1u) mx = fmaxf(mx, s[r]);
  return mx;
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
  const floatx16 s = exact_scores<T, D>(qreg, kbase, k_row_bytes, key0, n_keys, lane);
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
