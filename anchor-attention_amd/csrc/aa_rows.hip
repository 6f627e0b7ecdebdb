// Dense attention of any number of query rows over any number of keys on gfx950: the planning of the flash kernel's rows
// mode (aa_flash.hip) and the kernel that merges its key chunks.
//
// Why rows have a kernel of their own: library attention takes a ragged causal window only as an explicit boolean mask,
// and then multiplies, masks and soft-maxes the whole score matrix in float32 in memory.  1089 rows over 40001 keys with
// 32/8 heads of 128 took 18.7 ms that way and take 0.97 ms + 0.03 ms (combine) here, 0.7 PFLOP/s of scores and P.V; 777 rows
// over 777 keys took 403 us and take 22 us.  A left-padded batch of 3 x 2500 tokens with its boolean mask took 7.66 ms and
// takes 0.22 ms: the mask is packed to bits once, and tiles in which no row of a work-group sees a key are not visited.
// Probabilities were float32 there: each enters P.V as two 16-bit numbers (bf16: 16 bits of it; fp16: 22, formed with a
// factor that keeps small ones off the subnormals' grid, see kProbLog2).  That costs a second MFMA
// per V operand (with one: 0.80 ms, 20 us and 0.19 ms) and brings the error against float64 from up to 1.02 times that of
// library attention to the same (1.460e-3, 1.468e-3 with one, padded 3 x 1000, bf16).
#include <cmath>

#include "aa_common.h"
#include "aa_kernels.h"
#include "aa_nonfinite.h"

namespace aa {

// Merges the key chunks of rows mode: out = sum_c w_c acc_c / sum_c w_c l_c with w_c = exp2((m_c - max m) * scale).
// One work-group per 128-column block and 32-column piece of the head dimension; lane layout and order of the state are
// those of the flash kernel that wrote it, so every load moves one contiguous KiB per wave.  Bound by reading the state,
// which the flash kernel has just written (L2 / memory-side cache).
template <typename T, int D>
__global__ void __launch_bounds__(256) rows_combine_kernel(const FlashArgs p) {
  constexpr int kDB = D / 32;
  const int lane = threadIdx.x & 63, half = lane >> 5, c32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t id = blockIdx.x;
  const int db = id % kDB;  id /= kDB;
  const int block = take_remainder(id, p.by_cols, p.n_col_blocks);
  const int b = quotient(id, p.by_kv_heads), kvh = id - b * p.n_kv_heads;
  const int group = p.group, n_cols = p.n_rows * group;
  // the chunks that hold keys of this block (the others were not written)
  const int last_row = quotient(min(128 * block + 128, n_cols) - 1, p.by_group);
  const int tiles = min(p.causal_offset + last_row, p.n_ctx - 1) / 64 + 1;
  const int n_chunks = quotient(tiles + p.chunk_tiles - 1, p.by_chunks);
  const int64_t slot0 = ((((int64_t)b * p.n_kv_heads + kvh) * p.n_col_blocks + block) * p.n_chunks) * 4 + wave;
  const float scale = p.sm_scale * kLog2e;

  float m_all = -INFINITY;
#pragma unroll 4
  for (int c = 0; c < n_chunks; ++c) m_all = fmaxf(m_all, p.M[(slot0 + 4 * c) * 32 + c32]);
  floatx4 acc[4];
  float l_all;
  auto merge = [&](const float factor) __attribute__((always_inline)) {
    l_all = 0.f;
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) acc[rg] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int c = 0; c < n_chunks; ++c) {
      const int64_t slot = slot0 + 4 * c;
      const float m = p.M[slot * 32 + c32];
      const float w = m == -INFINITY ? 0.f : fast_exp2((m - m_all) * scale) * factor;  // (a chunk without a key of this row's)
      l_all += w * p.L[slot * 32 + c32];
      const float* af = p.acc_frag + (slot * kDB + db) * (4 * 256) + lane * 4;
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const floatx4 t = *reinterpret_cast<const floatx4*>(af + rg * 256);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[rg][e] += w * t[e];
      }
    }
  };
  merge(1.f);
  if (T::kProbLog2 == 0.f) {
    // bf16 chunks' sums are finite but may have probabilities above 1 in them (aa_nonfinite.h), and V so large that together they are not.
    // Then once more, divided by the power of two that the sum of the probabilities holds: exact, and no larger than V.
    float sum = 0.f;
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) sum += (acc[rg][0] + acc[rg][1]) + (acc[rg][2] + acc[rg][3]);
    if (__builtin_expect(__any(!is_finite(sum) && l_all > 1.f && is_finite(l_all)), 0))
      merge(l_all > 1.f && is_finite(l_all) ? __uint_as_float((254u << 23) - (__float_as_uint(l_all) & 0x7f800000u)) : 1.f);
  }
  const float inv = l_all == 0.f ? 0.f : 1.f / l_all;  // (masked mode: a row that sees no key gives 0)
  uint32_t w[4][2];
#pragma unroll
  for (int rg = 0; rg < 4; ++rg) {
    w[rg][0] = T::pack(acc[rg][0] * inv, acc[rg][1] * inv);
    w[rg][1] = T::pack(acc[rg][2] * inv, acc[rg][3] * inv);
  }
  // a lane holds columns 8*rg + 4*half .. +3 of the piece: the two halves of the wave trade register groups, so that each
  // lane stores whole 16-byte chunks (half 0 the even groups, half 1 the odd ones)
  const int col = 128 * block + 32 * wave + c32;
  const int row = quotient(min(col, n_cols - 1), p.by_group);
  uint16_t* op = p.out + b * p.o_sb + (int64_t)(kvh * group + min(col, n_cols - 1) - row * group) * p.o_sh + (int64_t)row * p.o_sn + 32 * db;
#pragma unroll
  for (int pr = 0; pr < 2; ++pr) {
    const uint32_t r0 = __shfl_xor(half ? w[2 * pr][0] : w[2 * pr + 1][0], 32, 64);
    const uint32_t r1 = __shfl_xor(half ? w[2 * pr][1] : w[2 * pr + 1][1], 32, 64);
    uint4 o;
    if (half == 0) o = uint4{w[2 * pr][0], w[2 * pr][1], r0, r1};
    else o = uint4{r0, r1, w[2 * pr + 1][0], w[2 * pr + 1][1]};
    if (col < n_cols) *reinterpret_cast<uint4*>(op + 8 * (2 * pr + half)) = o;
  }
}

hipError_t launch_rows_combine(FlashArgs a, hipStream_t stream) {
  set_heads(a);
  a.by_cols = fast_div(a.n_col_blocks);
  a.by_chunks = fast_div(a.chunk_tiles);
  const dim3 grid((uint32_t)a.batch * a.n_kv_heads * a.n_col_blocks * (a.head_dim / 32)), block(256);
  if (a.head_dim == 128) {
    if (a.dtype == 0) hipLaunchKernelGGL((rows_combine_kernel<Bf16, 128>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((rows_combine_kernel<F16, 128>), grid, block, 0, stream, a);
  } else {
    if (a.dtype == 0) hipLaunchKernelGGL((rows_combine_kernel<Bf16, 64>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((rows_combine_kernel<F16, 64>), grid, block, 0, stream, a);
  }
  return hipGetLastError();
}

// Masked mode: packs the byte mask of one column block's rows, 64 keys to a word, and notes for each 64-key tile whether any
// and whether every one of the rows sees it.  A work-group takes 1024 keys of the block's rows, a lane 16 of them; the four
// waves share the rows, eight loads in flight each.  Bound by the latency of its rounds of loads (32 rows each: one or two with heads
// in groups of four at most, four without groups): a mask is read once (rows that two column blocks share are packed twice, to the same words).  A row's last keys are read as its last 16
// and shifted, not byte by byte.  3 x 2500 x 2500: 32.1 us with a wave to a block's rows and a byte loop, 7.3 us now.
constexpr int kPackKeys = 1024;
__global__ void __launch_bounds__(256) mask_pack_kernel(const FlashArgs p, const uint8_t* mask, const int64_t mask_sb, const int64_t mask_sn) {
  __shared__ uint32_t seen[4][kPackKeys / 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int block = blockIdx.y, b = blockIdx.z;
  const int group = p.n_q_heads / p.n_kv_heads, n_cols = p.n_rows * group;
  const int row0 = 128 * block / group, row1 = (min(128 * block + 128, n_cols) - 1) / group;  // first and last row of the block
  const int key0 = blockIdx.x * kPackKeys + 16 * lane;
  const int tile = key0 / 64;
  const int from = max(min(key0, p.n_ctx - 16), 0);  // this lane's 16 bytes of a row, inside the row
  const int shift = min(key0 - from, 16);            // those that belong to the lane before; 16: the row ends before this lane
  const uint8_t* src = mask + b * mask_sb + from;
  uint64_t* words = const_cast<uint64_t*>(p.mask_words) + (int64_t)b * p.n_rows * p.mask_words_per_row;
  uint32_t any = 0u, all = 0xffffu;
  constexpr int kBatch = 8;
  for (int r0 = row0 + wave; r0 <= row1; r0 += 4 * kBatch) {
    uint32_t x[kBatch][4];
    // (past the last row: that row again, with the same result)
    if (p.n_ctx >= 16) {
#pragma unroll
      for (int j = 0; j < kBatch; ++j) __builtin_memcpy(x[j], src + (int64_t)min(r0 + 4 * j, row1) * mask_sn, 16);
    } else {
#pragma unroll
      for (int j = 0; j < kBatch; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const uint32_t byte = i < p.n_ctx ? (src + (int64_t)min(r0 + 4 * j, row1) * mask_sn)[i] : 0u;
          x[j][i >> 2] = (i & 3 ? x[j][i >> 2] : 0u) | byte << (8 * (i & 3));
        }
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int row = min(r0 + 4 * j, row1);
      uint32_t bits = 0u;
#pragma unroll
      for (int i = 0; i < 4; ++i) {  // bytes 0/1 -> four bits: the products meet at bits 24..27 without carries
        const uint32_t ones = (x[j][i] | (x[j][i] >> 4)) | ((x[j][i] | (x[j][i] >> 4)) >> 2);  // any bit of a byte counts as true
        bits |= ((((ones | (ones >> 1)) & 0x01010101u) * 0x01020408u) >> 24 & 0xfu) << (4 * i);
      }
      bits >>= shift;
      any |= bits;
      all &= bits;
      // four lanes make a word
      const uint32_t pair = bits | (__shfl_down(bits, 1, 64) << 16);
      const uint32_t high = __shfl_down(pair, 2, 64);
      if ((lane & 3) == 0 && tile < p.mask_words_per_row) words[(int64_t)row * p.mask_words_per_row + tile] = (uint64_t)pair | (uint64_t)high << 32;
    }
  }
  any |= __shfl_xor(any, 1, 64);
  any |= __shfl_xor(any, 2, 64);
  all &= __shfl_xor(all, 1, 64);
  all &= __shfl_xor(all, 2, 64);
  if ((lane & 3) == 0) seen[wave][lane >> 2] = any << 16 | all;
  __syncthreads();
  const int my_tile = blockIdx.x * (kPackKeys / 64) + threadIdx.x;
  if (threadIdx.x < kPackKeys / 64 && my_tile < p.mask_words_per_row) {
    any = all = seen[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      any |= seen[w][threadIdx.x];
      all &= seen[w][threadIdx.x];
    }
    const_cast<uint8_t*>(p.tile_flags)[((int64_t)b * p.n_col_blocks + block) * p.mask_words_per_row + my_tile] =
        (all & 0xffffu) == 0xffffu ? 2 : any >> 16 ? 1 : 0;
  }
}

hipError_t launch_mask_pack(const FlashArgs& a, const uint8_t* mask, int64_t mask_sb, int64_t mask_sn, hipStream_t stream) {
  const dim3 grid((a.n_ctx + kPackKeys - 1) / kPackKeys, a.n_col_blocks, a.batch);
  hipLaunchKernelGGL(mask_pack_kernel, grid, dim3(256), 0, stream, a, mask, mask_sb, mask_sn);
  return hipGetLastError();
}

// Sets the number of column blocks; the tiles that a unit's (a KV head's) last columns see.
static int set_columns(FlashArgs& a) {
  a.n_col_blocks = (a.n_rows * (a.n_q_heads / a.n_kv_heads) + 127) / 128;
  return (min(a.causal_offset + a.n_rows, a.n_ctx) + 63) / 64;
}
// column blocks that see a key of tile t: those whose last row is at least 64 t - causal_offset
static int blocks_at(const FlashArgs& a, const int t) {
  return a.n_col_blocks - (int)((int64_t)max(64 * t - a.causal_offset, 0) * (a.n_q_heads / a.n_kv_heads) / 128);
}
// tiles of a unit's work-groups
static int64_t unit_tiles(const FlashArgs& a, const int max_tiles) {
  const int all_see = min(a.causal_offset / 64 + 1, max_tiles);
  int64_t total = (int64_t)all_see * a.n_col_blocks;
  for (int t = all_see; t < max_tiles; ++t) total += blocks_at(a, t);
  return total;
}
constexpr int kMaxChunks = 64;

// How the keys of a rows-mode problem are cut into chunks: every number of chunks up to 64 is priced and the cheapest taken.
//
// Work-groups are dealt to the CUs in turn, the ones with the most tiles first, so the CU that gets the longest chain of tiles gets, 256
// work-groups on, its second one (head dimension 64: and a third) as long as the chip has room: a bf16 tile takes 1.1 us while a
// work-group is alone on its CU and 1.8 beside another (64: 0.8, 1.1 and 1.3 beside two).  A launch takes as long as that CU or
// as all tiles at the rate of a full chip, 0.9 us a tile and CU (64: 0.45) - the fourth powers are added, which lies between the larger and the sum - and
// a part of a chain for the uneven end of more than one round.  Several chunks cost one more launch and a write and a read
// of the state (64 KB per column block and chunk at head dimension 128).  fp16 has prices of its own: its probabilities need the running max, so that
// a tile of a work-group alone takes 1.2 us at head dimension 128.
//
// The bf16 prices were fitted to 192 sizes (20 to 5000 rows over up to 40000 keys, 2 to 32 KV heads in groups of 4 and 7, each with up to twelve
// numbers of chunks), the fp16 ones to the 2042 of 5 to 3000 rows and 1 to 4 prompts on which both are compared here.  The number taken is slower than the
// best of about ten measured ones by 1.0 % on average (98 of 100 within 11 %), fp16 0.7 (8) %, at 64 2.3 (27) and 1.4 (15) %, most of it where a
// call is so short that a second launch costs the host more than it gives the GPU.  (440 other sizes, some of them masked, on the kernel as it is since: 1.0, 1.1,
// 1.7 and 0.9 %.)  The form before, which had the longest chain or the rounds of a full chip at
// one price, came to 2.4, 1.2, 4.3 and 2.5 %: it did not know that a few work-groups more than CUs share them with the lightest ones (1194 rows,
// 28/4 heads of 128: 36.9 us in three chunks, 30.2 whole); 30 of the 4084 are more than 5 % slower than with it, by 14 % at most.  With the bf16 prices for
// fp16 those were 92 (22 %): 649 rows over 2890 keys, 32/8 heads of 128, 82.2 us in one chunk, 68.6 in three.
//
// A column block whose rows end later sees no fewer keys, so the blocks that reach a tile are counted in closed form and a plan costs the
// same whatever the rows: with a loop over the column blocks for every count it took the host 276 us for 32768 rows over 65536 keys
// and 1.1 ms for 131072 masked rows (32/8 heads), twice a call, and takes 4 us.
void plan_rows(FlashArgs& a) {
  const int max_tiles = set_columns(a), group = a.n_q_heads / a.n_kv_heads;
  const int64_t units = (int64_t)a.batch * a.n_kv_heads, total = unit_tiles(a, max_tiles);
  const bool wide = a.head_dim == 128;
  const int slots = wide ? 512 : 768;
  // us a tile; us a tile of the longest chain, a full chip's round, a merge and a MB of state
  struct Prices { double alone, beside_one, beside_two, full_chip, uneven_end, one_round, merge, merge_per_mb; };
  static const Prices kPrices[2][2] = {{{0.835, 1.105, 1.306, 0.448, 0.098, 0.244, 1.57, 0.467}, {1.07, 1.81, 0.0, 0.912, 0.616, 0.083, 2.65, 0.242}},
                                           {{0.87, 1.16, 1.27, 0.46, 0.10, 0.26, 2.5, 0.365}, {1.21, 1.61, 0.0, 0.88, 0.45, 0.083, 2.15, 0.23}}};
  const Prices& price = kPrices[a.dtype != 0][wide];
  const int64_t second = units <= 256 ? 256 / units : 1;  // the number, among a unit's work-groups, of the one that joins the first on its CU
  double best = 1e30;
  a.n_chunks = 1;
  a.chunk_tiles = max_tiles;
  const int n_min = a.mask_words_per_row > 0 ? (max_tiles + kMaskedTiles - 1) / kMaskedTiles : 1;
  for (int n = n_min; n <= kMaxChunks && n <= max_tiles; ++n) {
    const int len = (max_tiles + n - 1) / n, chunks = (max_tiles + len - 1) / len;
    int64_t wgs = 0;
    for (int c = 0; c < chunks; ++c) wgs += blocks_at(a, c * len);
    wgs *= units;
    // tiles of a unit's k-th work-group: latest column blocks first, chunk by chunk
    auto tiles_of = [&](const int64_t k) {
      if (k >= (int64_t)a.n_col_blocks * chunks) return 0;
      const int block = a.n_col_blocks - 1 - (int)(k % a.n_col_blocks), last_row = (int)(min(128 * (int64_t)block + 128, (int64_t)a.n_rows * group) - 1) / group;
      const int seen = min(a.causal_offset + last_row, a.n_ctx - 1) / 64 + 1;
      return max(0, min(seen - (int)(k / a.n_col_blocks) * len, len));
    };
    const int t0 = tiles_of(0), t1 = min(tiles_of(second), t0), t2 = wide ? 0 : min(tiles_of(2 * second), t1);
    const double chain = price.alone * (t0 - t1) + price.beside_one * (t1 - t2) + price.beside_two * t2;
    const double all = price.full_chip * (double)total * units / 256;
    const double c2 = chain * chain, a2 = all * all;
    double us = std::sqrt(std::sqrt(c2 * c2 + a2 * a2)) + (wgs > slots ? price.uneven_end * len : 0.0) + price.one_round * (double)wgs / slots;
    if (chunks > 1) us += price.merge + price.merge_per_mb * (double)wgs * 128 * a.head_dim * 8 / 1e6;
    if (us < best) {
      best = us;
      a.n_chunks = chunks;
      a.chunk_tiles = len;
    }
  }
}

// Beside anchor work-groups, which fill the chip and the end of the launch, the chunks only have to keep a chain of tiles from
// outlasting everything else: the fewest chunks whose tiles take no longer (head dimension 128: 1.3 us each, 64: 1.15) than all tiles of
// the launch on a full chip (per CU 0.9 us an anchor tile and 1.3 a rows tile, whose probabilities enter twice; 64: 0.5 and 0.72) or than
// the longest anchor work-group (1.0 us a tile, 64: 0.8).  That is one chunk, and no merge, for all but short prompts and few heads: on 56 sizes (prompts
// of 2080 to 40001 tokens) 0.2 % slower than the best of 1, 2, 3, 4 and 6 chunks on average, 3.4 % at worst.
void plan_rows_beside(FlashArgs& a, const FlashArgs& anchor) {
  const int max_tiles = set_columns(a);
  const bool wide = a.head_dim == 128;
  const int64_t s = anchor.big_block / 128, n_big = anchor.n_ctx / anchor.big_block;  // 128-row blocks of a big block
  const int64_t anchor_tiles = (n_big * s * (s + 1) + (n_big - 1) * 2 * s * s) * anchor.batch * anchor.n_q_heads;
  const double all = ((wide ? 0.9 : 0.5) * (double)anchor_tiles + (wide ? 1.3 : 0.72) * (double)(unit_tiles(a, max_tiles) * a.batch * a.n_kv_heads)) / 256;
  const double anchor_chain = (wide ? 1.0 : 0.8) * (double)((n_big > 1 ? 4 : 2) * s);
  const int longest = max((int)(fmax(all, anchor_chain) / (wide ? 1.3 : 1.15)), 1);
  const int n = min((max_tiles + longest - 1) / longest, kMaxChunks);
  a.chunk_tiles = (max_tiles + n - 1) / n;
  a.n_chunks = (max_tiles + a.chunk_tiles - 1) / a.chunk_tiles;
}

}  // namespace aa
