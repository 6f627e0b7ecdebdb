// Shared device/host helpers for the AnchorAttention gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace aa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.44269504f;  // the literal the operator's definition multiplies by

// ---- 16-bit element types --------------------------------------------------------------------
// The operator takes bf16 tensors (what its callers use) or fp16 tensors (which the definition also admits: every
// ".to(dtype)" of it then rounds to fp16).  A kernel is written once against one of these two descriptions of the
// element type: unpacking a pair from a dword, round-to-nearest-even packing, and the matching MFMA.
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// kProbLog2: where a probability p <= 1 is kept as two 16-bit numbers (its rounding and the rest), 2^kProbLog2 * p is formed
// instead; the sums of probabilities carry the same factor and it cancels in the quotient.  fp16 needs it: p and its rest lie
// on the grid of the subnormals, 2^-24, as soon as p is below 2^-14 - the keys that lose to an attention sink by ten
// nats.  2^15 * p (at most 32768) puts the rest's grid at 2^-39 of the sum's scale: the pair is off by 2^-22 of p down to
// p = 2^-18, by 2^-16 down to 2^-24 (17 nats below the largest), by 2^-11, a result's own rounding, at 2^-29 (20 nats).
struct Bf16 {
  typedef bf16x8 vec8;
  static constexpr float kProbLog2 = 0.f;
  static constexpr uint16_t kExponent = 0x7f80;  // its bits, all of them set in infinities and NaN
  static __device__ __forceinline__ float lo(uint32_t u) { return __uint_as_float(u << 16); }
  static __device__ __forceinline__ float hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
  static __device__ __forceinline__ float from16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
  // round-to-nearest-even float -> bf16, two at a time (v_cvt_pk_bf16_f32 on gfx950)
  static __device__ __forceinline__ uint32_t pack(float a, float b) {
    floatx2 f = {a, b};
    bf16x2 h = __builtin_convertvector(f, bf16x2);
    return *reinterpret_cast<uint32_t*>(&h);
  }
  // the pair that rounding to `packed` took from a and b: a - lo and b - hi, exact, one instruction each as dot products of the pair
  // with (-1, 0) and (0, -1).  (The pairs are hidden from the compiler, which encodes constants of this instruction wrongly.)
  // Unpacked and subtracted: 777 rows over 777 keys, 32/8 heads of 128, 20.9 us against 20.5; padded 3 x 2500 194.8 against 191.7.
  static __device__ __forceinline__ uint32_t pack_rest(float a, float b, uint32_t packed) {
    uint32_t minus_lo = 0x0000bf80u, minus_hi = 0xbf800000u;
    asm("" : "+s"(minus_lo));
    asm("" : "+s"(minus_hi));
    const bf16x2 p = *reinterpret_cast<const bf16x2*>(&packed);
    return pack(__builtin_amdgcn_fdot2_f32_bf16(p, *reinterpret_cast<const bf16x2*>(&minus_lo), a, false),
                __builtin_amdgcn_fdot2_f32_bf16(p, *reinterpret_cast<const bf16x2*>(&minus_hi), b, false));
  }
  static __device__ __forceinline__ float round(float a) { return lo(pack(a, 0.f)); }  // float -> nearest bf16 -> float
  // (a * b).to(bf16) as the operator's definition compiles: a float32 product, then the rounding
  static __device__ __forceinline__ float round_product(float a, float b) { return round(a * b); }
  static __device__ __forceinline__ floatx16 mfma(vec8 a, vec8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

struct F16 {
  typedef f16x8 vec8;
  static constexpr float kProbLog2 = 15.f;
  static constexpr uint16_t kExponent = 0x7c00;
  static __device__ __forceinline__ float lo(uint32_t u) { return (float)(*reinterpret_cast<f16x2*>(&u))[0]; }
  static __device__ __forceinline__ float hi(uint32_t u) { return (float)(*reinterpret_cast<f16x2*>(&u))[1]; }
  static __device__ __forceinline__ float from16(uint16_t h) { return lo((uint32_t)h); }
  // round-to-nearest-even float -> fp16, two at a time (v_cvt_pk_f16_f32 on gfx950); overflow gives infinity
  static __device__ __forceinline__ uint32_t pack(float a, float b) {
    floatx2 f = {a, b};
    f16x2 h = __builtin_convertvector(f, f16x2);
    return *reinterpret_cast<uint32_t*>(&h);
  }
  // (as fused operations, which take 16-bit operands as they are; the factor is hidden from the compiler, which makes a conversion
  // and a subtraction of it)
  static __device__ __forceinline__ uint32_t pack_rest(float a, float b, uint32_t packed) {
    float minus_one = -1.f;
    asm("" : "+s"(minus_one));
    return pack(__builtin_fmaf(lo(packed), minus_one, a), __builtin_fmaf(hi(packed), minus_one, b));
  }
  static __device__ __forceinline__ float round(float a) { return lo(pack(a, 0.f)); }
  // (a * b).to(fp16) as the operator's definition compiles: ONE rounding of the exact product (the multiply and the
  // cast become a single mixed-precision instruction).  Written out so that it does not depend on what this compiler
  // fuses: the product is exact in double; it is brought to float32 with round-to-odd, after which the
  // round-to-nearest-even to fp16 is the correct rounding of the exact value.
  static __device__ __forceinline__ float round_product(float a, float b) {
    const double d = (double)a * (double)b;
    float f = (float)d;
    const double back = (double)f;
    if (back != d) {  // inexact (also: overflow to infinity)
      uint32_t u = __float_as_uint(f);
      if ((u & 1u) == 0u) {  // even: the odd neighbour on d's side
        const bool negative = (u >> 31) != 0u, larger = d > back;
        u = (negative != larger) ? u + 1u : u - 1u;
      }
      f = __uint_as_float(u);
    }
    return round(f);
  }
  static __device__ __forceinline__ floatx16 mfma(vec8 a, vec8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// 2^(x * scale + kProbLog2): a probability that is to be kept as two 16-bit numbers (bf16: without the addition of 0)
template <typename T>
__device__ __forceinline__ float prob_exp2(float x, float scale) {
  return fast_exp2(T::kProbLog2 != 0.f ? __builtin_fmaf(x, scale, T::kProbLog2) : x * scale);
}

// Work-group barrier for LDS hand-over only: waits for this wave's LDS traffic, then synchronises.
// Unlike __syncthreads() it does not wait for outstanding global loads, so prefetches issued before
// the barrier stay in flight across it.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

typedef __attribute__((address_space(3))) char lds_char;
__device__ __forceinline__ uint32_t lds_addr(const void* p) { return (uint32_t)(uintptr_t)(lds_char*)p; }

// 64 lanes x 16 bytes, global -> LDS without passing through registers: lane L's bytes land at
// lds_dst + 16*L (lds_dst is wave-uniform and travels in M0).  Completion is tracked by vmcnt.
__device__ __forceinline__ void load16_to_lds(const char* base, const uint32_t byte_off, const uint32_t lds_dst) {
  // the LDS base is bound to M0 by the constraint, so the compiler knows that M0 is written here; the nop covers the
  // wait state an LDS-DMA instruction needs after a scalar write of M0 (the compiler does not look inside the asm)
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "{m0}"(lds_dst), "v"(byte_off), "s"(base) : "memory");
}

// value held by the lane 32 positions away (the two halves of a wave share MFMA columns)
__device__ __forceinline__ float xor32(float v) { return __shfl_xor(v, 32, 64); }

// max of a value and its counterpart 32 lanes away, without a trip through LDS: v_permlane32_swap hands every
// lane the lower half's value (result 0) and the upper half's value (result 1)
__device__ __forceinline__ float max_with_other_half(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// The share of selected keys, sum(counts[0 .. n)) * inverse, by one work-group of 256 threads: a few KB, bound by the latency of
// a round trip or two.  `part`: four words of LDS.  (As a launch of its own 5.8 us of the 198 us of the operator on 4096 tokens with
// 32/8 heads of 128, and the framework's sum and division, four launches, 14 us.)
__device__ __forceinline__ void store_ratio(const float x, float* ratio, float* ratio_host) {
  *ratio = x;
  if (ratio_host != nullptr) __hip_atomic_store(ratio_host, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// The same by all work-groups of a launch, each with the keys that it has selected (`mine`, of its first thread): one 64-bit atomic each, work-groups that
// have come in the upper bits and keys in the lower 44.  The last one stores the ratio.  The number is the atomic's own, so nothing else has to be ordered.
__device__ __forceinline__ void add_selected(const uint32_t mine, uint64_t* selected, const float inverse, float* ratio, float* ratio_host) {
  constexpr uint64_t kOne = 1ull << 44;
  const uint64_t sum = __hip_atomic_fetch_add(selected, kOne + mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + (kOne + mine);
  if (sum >> 44 == gridDim.x) store_ratio((float)(int64_t)(sum & (kOne - 1)) * inverse, ratio, ratio_host);
}

__device__ __forceinline__ void sum_counts(const int32_t* counts, const int64_t n, const float inverse, float* ratio, float* ratio_host,
                                           int64_t* part) {
  int64_t sum = 0;
  for (int64_t i = threadIdx.x; i < n; i += 256) sum += counts[i];
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor((long long)sum, d, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) store_ratio((float)(part[0] + part[1] + part[2] + part[3]) * inverse, ratio, ratio_host);
}

// ---- division by a number that the host knows --------------------------------------------------
// Every work-group finds its place by some ten divisions, of 150 to 200 clocks one after the other where the compiler divides by a number it does
// not know, and those of rows have eight more beside their stores; with the reciprocal from the host a division is a multiplication, two
// additions and two shifts.  (Granlund and Montgomery, Division by invariant integers using multiplication: exact for all 32-bit numbers.)
// 32/8 heads of 128: 777 rows 20.1 -> 19.85 us, padded 2 x 1500 63.6 -> 62.3 and 3 x 2500 186 -> 184.4, a decode step over 33001 keys 28.65 -> 28.25;
// 131072 tokens 7343 -> 7328.
//
// A reciprocal costs the host a 64-bit division, so a launch forms those that its kernel divides by and no others.  (With thirteen
// of them for every launch short calls took 0.1 to 0.2 us longer than without any: decode steps over 300 to 9000 keys 15 to 21 us, 0.8 % on average; 0.1 % now.)
struct FastDiv {
  uint32_t mul, shifts;  // two shifts, 0 or 1 in the lower five bits and one in the upper 24
};
inline FastDiv fast_div(const uint32_t d) {  // d >= 1
  const uint32_t bits = d > 1 ? 32 - (uint32_t)__builtin_clz(d - 1) : 0;
  return {(uint32_t)((((1ull << bits) - d) << 32) / d + 1), bits > 0 ? 1u | (bits - 1) << 8 : 0u};
}
__host__ __device__ __forceinline__ uint32_t quotient(const uint32_t n, const FastDiv& f) {
  const uint32_t t = (uint32_t)((uint64_t)n * f.mul >> 32);
  return (t + ((n - t) >> (f.shifts & 31u))) >> (f.shifts >> 8);
}
// n divided by the divisor of f; n becomes the quotient, the remainder is returned
__host__ __device__ __forceinline__ uint32_t take_remainder(uint32_t& n, const FastDiv& f, const uint32_t d) {
  const uint32_t q = quotient(n, f), r = n - q * d;
  n = q;
  return r;
}

// ---- geometry --------------------------------------------------------------------------------
// Index lists are packed per (batch, query head): big block bb can select at most
// cap(bb) = bb*S - 2*bs keys (candidates are [bs, bb*S - bs)), and its list starts at
// tri(bb) = sum_{x<bb} cap(x) entries into the head's slab.
__host__ __device__ inline int64_t coords_tri(int64_t bb, int64_t S, int64_t bs) {
  return bb <= 1 ? 0 : S * (bb - 1) * bb / 2 - 2 * bs * (bb - 1);
}

// XCD-aware work-group renumbering.  Consecutive hardware work-group ids go round-robin over the 8 XCDs (each
// with its own L2).  The work consists of `n_units` units (a KV head of one batch element) of `per_unit`
// work-groups each, ordered heaviest first inside a unit; work-groups of one unit read the same K/V rows or pooled
// queries.  Gives (unit, idx in the unit) such that
//   n_units % 8 == 0 : every XCD owns n_units / 8 whole units, every eighth one: the units of one batch element, whose work
//                      differs from another's where prompts are padded, are spread over the XCDs;
//   8 % n_units == 0 : s = 8 / n_units XCDs share a unit and take its rows alternately (row = idx / inner, the
//                      `inner` work-groups of a row stay together), so that each gets the same mix of heavy and light;
//   otherwise        : the hardware order is kept.
// The host makes the choice and the reciprocal.  `abreast`: an XCD takes its units (in the last case: all XCDs all units) side by side, the heaviest of each first, instead of one
// after the other, so that the launch does not end with the heaviest work-groups of its last unit.
struct Deal {
  enum Kind : uint32_t { kInTurn, kOwnUnits, kSharedUnits, kAbreast, kAbreastAll } kind;
  uint32_t n; FastDiv by_n;  // work-groups of a unit (in turn, own units) or of a row (shared units); units of an XCD or all units (abreast)
  uint32_t share_log;        // (shared units) log2 of the XCDs that share one
  uint32_t turns;            // (abreast) an XCD's units begin one further on every 32 work-groups
};
inline Deal make_deal(uint32_t n_units, uint32_t per_unit, uint32_t inner, bool abreast) {
  Deal d = {Deal::kInTurn, per_unit, {}, 0, 0};
  const bool even = (uint64_t)n_units * per_unit % 8 == 0;
  if (abreast) {
    d.kind = !even || n_units % 8 != 0 ? Deal::kAbreastAll : Deal::kAbreast;
    d.n = d.kind == Deal::kAbreast ? n_units / 8 : n_units;
    // (the XCD's 32 CUs are filled in turn: without the rotation a number of units that divides 32 ties a CU to a unit, and
    // units differ in weight: two prompts of 3900, one padded, 239 us one after the other, 280 without it and 239 with it)
    d.turns = 32 % d.n == 0;
  } else if (even && n_units % 8 == 0) {
    d.kind = Deal::kOwnUnits;
  } else if (even && 8 % n_units == 0 && (per_unit / inner) % (8 / n_units) == 0) {
    d.kind = Deal::kSharedUnits;
    d.n = inner;
    for (uint32_t s = 8 / n_units; s > 1; s /= 2) ++d.share_log;
  }
  d.by_n = fast_div(d.n);
  return d;
}
__host__ __device__ __forceinline__ void dealt(const Deal& d, const uint32_t wg, uint32_t& unit, uint32_t& index) {
  const uint32_t xcd = wg % 8u, k = wg / 8u;
  uint32_t n = d.kind == Deal::kInTurn || d.kind == Deal::kAbreastAll ? wg : k;
  if (d.kind == Deal::kAbreast && d.turns) n += k / 32u;
  const uint32_t r = take_remainder(n, d.by_n, d.n);
  if (d.kind == Deal::kOwnUnits) {
    unit = n * 8u + xcd;
    index = r;
  } else if (d.kind == Deal::kSharedUnits) {
    unit = xcd >> d.share_log;
    index = ((n << d.share_log) + (xcd & ((1u << d.share_log) - 1u))) * d.n + r;
  } else if (d.kind == Deal::kAbreast) {
    unit = r * 8u + xcd;
    index = quotient(k, d.by_n);
  } else {
    unit = d.kind == Deal::kAbreastAll ? r : n;
    index = d.kind == Deal::kAbreastAll ? n : r;
  }
}

// ---- error plumbing (host) -------------------------------------------------------------------
enum Status : int {
  kOk = 0,
  kBadArgument = 1,   // null pointer, non-positive size, inconsistent head counts
  kUnsupported = 2,   // a size the kernels are not written for (head_dim, block_size, step)
  kMisaligned = 3,    // pointer or stride breaks the 16-byte row alignment the loads assume
  kLaunchFailed = 4,  // the HIP runtime refused the launch
};
void set_error(const char* fmt, ...);

}  // namespace aa
