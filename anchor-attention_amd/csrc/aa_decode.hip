// Attention of a few query rows over a long key/value cache on gfx950 (decode steps): at most 32 (query row, head of the
// group) columns per KV head.
//
// Bound by reading K and V once.  The keys of a (batch, KV head) unit are cut into chunks, one work-group each, so that
// about one work-group per CU is at work; inside a work-group each of the four waves (or the only one: many units with short
// caches) streams its own 32-key tiles (tile t of the chunk to wave t % 4) through two private LDS slots filled by LDS-DMA,
// with no barrier until the end: a wave waits for its own loads only, and a CU has up to 128 KB in flight (head dimension
// 128).  All heads of a group are columns
// of the same products, so K and V are read once per KV head.  The arithmetic is that of the flash kernel's rows mode
// (S^T = K Q^T with the scores scaled in float32, online soft-max, O^T += V^T P^T); the waves' states are merged
// through LDS, the chunks' by decode_combine_kernel.
//
// (P enters the product as two 16-bit numbers, its rounding and the rest, as in the rows mode: 0.5 us.)
//
// One row, 32/8 heads of 128, 33001 keys (135 MB): 26.3 us = 5.1 TB/s, the rate of a large copy, and 4.1 us for the merge.
// The rows mode, which moves the state of 128 columns through its workspace, took 30.1 + 15.0 us; library attention, one
// work-group per head, 1164 us.
#include "aa_common.h"
#include "aa_kernels.h"
#include "aa_nonfinite.h"

namespace aa {

typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef short shortx8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

constexpr int kDecCols = 32;       // columns of a unit: query rows x heads of the group
constexpr int kDecTile = 32;       // keys a wave takes at a time
constexpr int kDecMaxChunk = 8192; // keys of a chunk (masked: the chunk's mask bits live in LDS)

template <typename T, int D, bool MASKED, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) decode_kernel(const FlashArgs p) {
  typedef typename T::vec8 vec8;
  typedef __attribute__((address_space(3))) vec8 lds_vec8;
  constexpr int kKS = D / 16, kDB = D / 32;
  constexpr int kPitch = 2 * D;                   // bytes of a row in LDS
  constexpr int kChunks = D / 8;                  // 16-byte chunks of a row
  constexpr int kRowsPerLoad = 64 / kChunks;      // rows one load instruction brings
  constexpr int kLoads = kDecTile / kRowsPerLoad; // load instructions of a K (or V) tile
  constexpr int kTile = kDecTile * kPitch;        // bytes of a K (or V) tile
  constexpr int kAccPitch = D + 4;                // floats of a column's accumulator when the waves are merged
  static_assert(kDecCols * kAccPitch * 4 <= 4 * kTile, "the waves' accumulators fit where their tiles were");
  // tiles by wave, slot and K/V.  (A single wave with a single tile is given one slot, see launch_decode_for)
  __shared__ __attribute__((aligned(16))) char fixed[WAVES > 1 ? WAVES * 4 * kTile : 16];
  extern __shared__ __attribute__((aligned(16))) char sized[];
  char* const tiles = WAVES > 1 ? fixed : sized;
  __shared__ float stats[2][WAVES][kDecCols];
  __shared__ uint64_t seen[MASKED ? kDecMaxChunk / 64 : 1];

  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, c32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int unit = quotient(blockIdx.x, p.by_chunks), chunk = blockIdx.x - unit * p.n_chunks;
  const int b = quotient(unit, p.by_kv_heads), kvh = unit - b * p.n_kv_heads;
  const int group = p.group, n_cols = p.n_rows * group;
  const int key_lo = chunk * p.chunk_tiles * kDecTile, key_hi = min(key_lo + p.chunk_tiles * kDecTile, p.n_ctx);
  const int n_tiles = (key_hi - key_lo + kDecTile - 1) / kDecTile;  // at least one: the host cuts the chunks so

  const char* kbase = reinterpret_cast<const char*>(p.k + b * p.k_sb + kvh * p.k_sh);
  const char* vbase = reinterpret_cast<const char*>(p.v + b * p.v_sb + kvh * p.v_sh);
  const uint32_t k_row = (uint32_t)p.k_sn * 2u, v_row = (uint32_t)p.v_sn * 2u;

  // 16-byte chunks are swizzled with the row, on the load side: K for row-per-lane 16-byte reads, V for transposing reads
  auto k_slot = [](const int row, const int c) { return D == 128 ? c ^ (row & 15) : c ^ ((row >> 1) & 7); };
  auto v_slot = [](const int row, const int c) { return D == 128 ? c ^ ((row & 7) << 1) : c ^ (((row >> 1) & 1) << 2); };
  auto issue = [&](const int t, const int slot) __attribute__((always_inline)) {
    const int key0 = key_lo + t * kDecTile, left = key_hi - key0;
    const char* kb = kbase + (uint64_t)(uint32_t)key0 * k_row;
    const char* vb = vbase + (uint64_t)(uint32_t)key0 * v_row;
    const uint32_t dst = lds_addr(tiles) + (2 * wave + slot) * (2 * kTile);
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int row = j * kRowsPerLoad + lane / kChunks;
      const uint32_t r = (uint32_t)min(row, left - 1);  // rows past the last key repeat it and are masked
      load16_to_lds(kb, __umul24(r, k_row) + 16u * k_slot(row, lane % kChunks), dst + j * 1024);
    }
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int row = j * kRowsPerLoad + lane / kChunks;
      const uint32_t r = (uint32_t)min(row, left - 1);
      load16_to_lds(vb, __umul24(r, v_row) + 16u * v_slot(row, lane % kChunks), dst + kTile + j * 1024);
    }
  };

  if (MASKED) {  // the chunk's mask bits, 64 keys to a word (a single row: the same for every column)
    const uint8_t* m = p.mask_bytes + b * p.mask_sb + key_lo;
    for (int i = 64 * wave; i < key_hi - key_lo; i += 64 * WAVES) {
      const uint64_t w = __ballot(i + lane < key_hi - key_lo && m[i + lane] != 0);
      if (lane == 0) seen[i / 64] = w;
    }
    __syncthreads();
  }
  auto tile_bits = [&](const int t) {
    return MASKED ? (uint32_t)(__builtin_amdgcn_readfirstlane(reinterpret_cast<const uint32_t*>(seen)[t])) : ~0u;
  };
  auto next_tile = [&](int t) {  // this wave's next tile in which a key is seen
    for (t += WAVES; MASKED && t < n_tiles && tile_bits(t) == 0u;) t += WAVES;
    return t;
  };

  int t = next_tile(wave - WAVES), t_next = n_tiles;
  if (t < n_tiles) {
    issue(t, 0);
    t_next = next_tile(t);
    if (t_next < n_tiles) issue(t_next, 1);
  }

  const int my_col = min(c32, n_cols - 1), my_row = quotient(my_col, p.by_group);
  const int my_last_key = MASKED ? p.n_ctx - 1 : min(p.causal_offset + my_row, p.n_ctx - 1);
  const int first_last_key = __builtin_amdgcn_readfirstlane(my_last_key);
  vec8 qreg[kKS];
  {
    const uint16_t* qr = p.q + b * p.q_sb + (int64_t)(kvh * group + my_col - my_row * group) * p.q_sh + (int64_t)my_row * p.q_sn + 8 * half;
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks) qreg[ks] = *reinterpret_cast<const vec8*>(qr + 16 * ks);
  }
  const float scale = p.sm_scale * kLog2e;
  float m_run = -INFINITY, l_run = 0.f;
  floatx16 acc[kDB];
#pragma unroll
  for (int db = 0; db < kDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;

  // LDS offsets inside a tile, as in the flash kernel: K row c32, chunk 2*ks + half; V by transposing reads
  const uint32_t tile0 = lds_addr(tiles) + wave * (4 * kTile);
  uint32_t k_rd[kKS], v_rd[kDB];
#pragma unroll
  for (int ks = 0; ks < kKS; ++ks) k_rd[ks] = tile0 + c32 * kPitch + 16 * k_slot(c32, 2 * ks + half);
  {
    const int r0 = 4 * half + ((lane & 15) >> 2), y0 = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
#pragma unroll
    for (int db = 0; db < kDB; ++db) v_rd[db] = tile0 + kTile + r0 * kPitch + 16 * v_slot(r0, 4 * db + y0) + 8 * (lane & 1);
  }

  int slot = 0;
  while (t < n_tiles) {
    // loads land in order: with the next tile's behind them, this tile's have landed when only those are outstanding
    if (t_next < n_tiles) {
      if (kLoads == 8) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const uint32_t off = slot * (2 * kTile);
    floatx16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks) s = T::mfma(*(const lds_vec8*)(uintptr_t)(k_rd[ks] + off), qreg[ks], s);
    const int key0 = key_lo + t * kDecTile;
    if (MASKED) {
      const uint32_t bits = tile_bits(t) >> (4 * half);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (!((bits >> (8 * (r >> 2) + (r & 3))) & 1u)) s[r] = -INFINITY;
    } else if (key0 + kDecTile - 1 > first_last_key) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (key0 + 8 * (r >> 2) + 4 * half + (r & 3) > my_last_key) s[r] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    const float m_new = fmaxf(m_run, max_with_other_half(mx));
    const float m_base = m_new == -INFINITY ? 0.f : m_new;  // (no key of this column's so far)
    if (__any(m_new > m_run)) {
      const float alpha = fast_exp2((m_run - m_base) * scale);
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < kDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
      m_run = m_new;
    }
    u32x4 pw[2], pw_rest[2];  // P^T and what its rounding left, both 16 bits wide
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        e[i] = prob_exp2<T>(s[4 * c + i] - m_base, scale);
        l_run += e[i];
      }
      pw[c >> 1][2 * (c & 1) + 0] = T::pack(e[0], e[1]);
      pw[c >> 1][2 * (c & 1) + 1] = T::pack(e[2], e[3]);
      // (unpacked and subtracted, not T::pack_rest: its longer latency shows in the chain of a wave alone, 20.2 us against 19.8 for
      // 33001 keys with 32/8 heads of 64)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t w = pw[c >> 1][2 * (c & 1) + i];
        pw_rest[c >> 1][2 * (c & 1) + i] = T::pack(e[2 * i] - T::lo(w), e[2 * i + 1] - T::hi(w));
      }
    }
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int db = 0; db < kDB; ++db) {
        const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(uintptr_t)(v_rd[db] + off + 16 * st * kPitch));
        const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(uintptr_t)(v_rd[db] + off + (16 * st + 8) * kPitch));
        const shortx8 a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        acc[db] = T::mfma(*reinterpret_cast<const vec8*>(&a), *reinterpret_cast<const vec8*>(&pw[st]), acc[db]);
        acc[db] = T::mfma(*reinterpret_cast<const vec8*>(&a), *reinterpret_cast<const vec8*>(&pw_rest[st]), acc[db]);
      }
    const int t_after = t_next < n_tiles ? next_tile(t_next) : n_tiles;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this slot has been read
    if (t_after < n_tiles) issue(t_after, slot);
    t = t_next;
    t_next = t_after;
    slot ^= 1;
  }

  if (__builtin_expect(__any(is_nan(sum_of_all(acc)) && !is_nan(l_run)), 0)) {
    // V holds infinities or NaN: the wave's sums once more (see aa_nonfinite.h)
    const float m_base = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
    for (t = next_tile(wave - WAVES); t < n_tiles; t = next_tile(t)) {
      const int key0 = key_lo + t * kDecTile, count = my_last_key + 1 - key0;
      const uint32_t seen = MASKED ? tile_bits(t) : count >= 32 ? ~0u : count <= 0 ? 0u : (1u << count) - 1u;
      exact_pv_tile<T, D>(acc, qreg, kbase, vbase, k_row, v_row, key0, key_hi, seen, m_base, scale, lane);
    }
  }

  // ---- the waves' states -> one ------------------------------------------------------------------
  const float l_tot = l_run + xor32(l_run);
  if (half == 0) {
    stats[0][wave][c32] = m_run;
    stats[1][wave][c32] = l_tot;
  }
  __syncthreads();  // (everyone is done with the tiles: the accumulators take their place)
  float* accs = reinterpret_cast<float*>(tiles);
  if (c32 < n_cols) {
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        floatx4 x;
#pragma unroll
        for (int c = 0; c < 4; ++c) x[c] = acc[db][4 * rg + c];
        *reinterpret_cast<floatx4*>(accs + (wave * kDecCols + c32) * kAccPitch + 32 * db + 8 * rg + 4 * half) = x;
      }
  }
  __syncthreads();
  for (int i = tid; i < n_cols * (D / 4); i += 64 * WAVES) {
    const int col = i / (D / 4), d = 4 * (i % (D / 4));
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) m = fmaxf(m, stats[0][w][col]);
    float l = 0.f;
    floatx4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float mw = stats[0][w][col];
      const float f = mw == -INFINITY ? 0.f : fast_exp2((mw - m) * scale);
      l += f * stats[1][w][col];
      const floatx4 y = *reinterpret_cast<const floatx4*>(accs + (w * kDecCols + col) * kAccPitch + d);
#pragma unroll
      for (int c = 0; c < 4; ++c) x[c] += f * y[c];
    }
    if (p.n_chunks == 1) {
      const float inv = l == 0.f ? 0.f : 1.f / l;
      const int row = quotient(col, p.by_group);
      uint16_t* op = p.out + b * p.o_sb + (int64_t)(kvh * group + col - row * group) * p.o_sh + (int64_t)row * p.o_sn + d;
      *reinterpret_cast<uint2*>(op) = uint2{T::pack(x[0] * inv, x[1] * inv), T::pack(x[2] * inv, x[3] * inv)};
    } else {
      const int64_t at = ((int64_t)unit * p.n_chunks + chunk) * n_cols + col;
      *reinterpret_cast<floatx4*>(p.acc_out + at * D + d) = x;
      if (d == 0) {
        p.M_out[at] = m;
        p.L_out[at] = l;
      }
    }
  }
}

// Merges the chunks of one column per work-group: the weights first, then eight groups of D/4 lanes each add up every
// eighth chunk.  A few KB per column out of the L2: bound by its two dependent rounds of loads.
template <typename T, int D>
__global__ void __launch_bounds__(256) decode_combine_kernel(const FlashArgs p) {
  constexpr int kLanes = D / 4, kParts = 256 / kLanes;
  __shared__ float weight[kDecMaxChunks];
  __shared__ float red[2][4];
  __shared__ floatx4 part[kParts][kLanes];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int group = p.group, n_cols = p.n_rows * group;
  const int unit = quotient(blockIdx.x, p.by_cols), col = blockIdx.x - unit * n_cols;
  const int64_t at0 = (int64_t)unit * p.n_chunks * n_cols + col;
  const float scale = p.sm_scale * kLog2e;
  // (at most 256 chunks: one per thread)
  const float m = tid < p.n_chunks ? p.M[at0 + (int64_t)tid * n_cols] : -INFINITY;
  const float l = tid < p.n_chunks ? p.L[at0 + (int64_t)tid * n_cols] : 0.f;
  float x = m;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) x = fmaxf(x, __shfl_xor(x, d, 64));
  if (lane == 0) red[0][wave] = x;
  __syncthreads();
  const float m_all = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
  const float w = m == -INFINITY ? 0.f : fast_exp2((m - m_all) * scale);
  weight[tid] = w;
  float y = w * l;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) y += __shfl_xor(y, d, 64);
  if (lane == 0) red[1][wave] = y;
  __syncthreads();
  const int g = tid / kLanes, d4 = tid % kLanes;
  floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int c = g; c < p.n_chunks; c += kParts) {
    const floatx4 v = *reinterpret_cast<const floatx4*>(p.acc_frag + (at0 + (int64_t)c * n_cols) * D + 4 * d4);
    const float f = weight[c];
#pragma unroll
    for (int e = 0; e < 4; ++e) sum[e] += f * v[e];
  }
  part[g][d4] = sum;
  __syncthreads();
  if (tid < kLanes) {
#pragma unroll
    for (int i = 1; i < kParts; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] += part[i][tid][e];
    const float l_all = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    const float inv = l_all == 0.f ? 0.f : 1.f / l_all;
    const int b = quotient(unit, p.by_kv_heads), kvh = unit - b * p.n_kv_heads, row = quotient(col, p.by_group);
    uint16_t* op = p.out + b * p.o_sb + (int64_t)(kvh * group + col - row * group) * p.o_sh + (int64_t)row * p.o_sn + 4 * tid;
    *reinterpret_cast<uint2*>(op) = uint2{T::pack(sum[0] * inv, sum[1] * inv), T::pack(sum[2] * inv, sum[3] * inv)};
  }
}

// Up to 32 columns are one MFMA's; from 33 on the rows mode, which shares a K/V tile among four waves of 32 columns, is the
// one that reads K and V once.  With a mask only a single row: its bits are the same for all columns.
bool decode_takes(int n_rows, int group, bool masked) { return n_rows * (int64_t)group <= kDecCols && (!masked || n_rows == 1); }

// One work-group per CU (256; head dimension 64, whose tiles are half as large: two) as far as the units allow, each with
// at least 256 keys - a wave's two tiles - and one up to 640 keys, below which the merge costs more than the reading (8 to 64 units: 384
// keys 8.2 us against 10.1 in two chunks, 512 9.6 against 10.5, 640 10.8 against 11.5, 768 12.0 against 11.3 in three).
//
// A work-group is four waves, whose tiles fill a CU's LDS, or a single one.  Four leave the CU to one unit, most of whose time goes
// by in starting, waiting for the first tile and merging, as soon as the units outnumber the CUs; of the single waves five (64:
// ten; nine and eighteen where there is one tile) share it.  8192 units of head dimension 128, one head each: 32 keys 118 us
// with four waves and 26 with one (library attention, which took such steps before: 72, and 16 keys 121, 22 and 19), 128 keys 159 and 98, 512 391 and
// 385, 1024 711 and 726; of 64: 32 keys 44 and 15, 192 79 and 75, 256 95 and 100.  256 units of 128: 64 keys 5.3 and 6.1, 32 keys 5.3 and 4.8.
void plan_decode(FlashArgs& a) {
  const int units = a.batch * a.n_kv_heads, slots = a.head_dim == 128 ? 256 : 512;
  int n = slots / units;
  n = n > (a.n_ctx + 255) / 256 ? (a.n_ctx + 255) / 256 : n;
  n = n > kDecMaxChunks ? kDecMaxChunks : n;
  if (a.n_ctx <= 640) n = 1;
  const int least = (a.n_ctx + kDecMaxChunk - 1) / kDecMaxChunk;
  n = n < least ? least : n;
  const int tiles = (a.n_ctx + kDecTile - 1) / kDecTile;
  a.chunk_tiles = (tiles + n - 1) / n;
  a.n_chunks = (tiles + a.chunk_tiles - 1) / a.chunk_tiles;
  a.n_col_blocks = 1;
  a.decode_waves = tiles == 1 || (units > slots && a.n_ctx <= (a.head_dim == 128 ? 512 : 192)) ? 1 : 4;
}

template <typename T, int D>
static void launch_decode_for(const FlashArgs& a, hipStream_t stream) {
  const int units = a.batch * a.n_kv_heads, group = a.n_q_heads / a.n_kv_heads;
  const dim3 grid((uint32_t)units * a.n_chunks), block(256);
  if (a.decode_waves == 1) {
    // LDS for one tile where there is one (at least what the accumulators take): nine work-groups on a CU instead of five
    const int tile = kDecTile * 2 * D, accs = kDecCols * (D + 4) * 4;
    const size_t lds = a.n_ctx > kDecTile ? 4 * tile : 2 * tile > accs ? 2 * tile : accs;
    if (a.mask_bytes) hipLaunchKernelGGL((decode_kernel<T, D, true, 1>), grid, dim3(64), lds, stream, a);
    else hipLaunchKernelGGL((decode_kernel<T, D, false, 1>), grid, dim3(64), lds, stream, a);
  } else {
    if (a.mask_bytes) hipLaunchKernelGGL((decode_kernel<T, D, true, 4>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((decode_kernel<T, D, false, 4>), grid, block, 0, stream, a);
  }
  if (a.n_chunks > 1) hipLaunchKernelGGL((decode_combine_kernel<T, D>), dim3((uint32_t)units * a.n_rows * group), block, 0, stream, a);
}

hipError_t launch_decode(FlashArgs& a, hipStream_t stream) {
  set_heads(a);
  a.by_chunks = fast_div(a.n_chunks);
  a.by_cols = fast_div((uint32_t)a.n_rows * a.group);  // (the columns are one block, and each is merged by a work-group)
  if (a.head_dim == 128) {
    if (a.dtype == 0) launch_decode_for<Bf16, 128>(a, stream);
    else launch_decode_for<F16, 128>(a, stream);
  } else {
    if (a.dtype == 0) launch_decode_for<Bf16, 64>(a, stream);
    else launch_decode_for<F16, 64>(a, stream);
  }
  return hipGetLastError();
}

}  // namespace aa
