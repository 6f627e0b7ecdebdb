// MFMA flash-attention core for gfx950, used five ways:
//   kAnchor : stage 1 - windowed causal attention over [0,S) U [bb*S, r]; emits M, L, Acc
//   kSparse : stage 3 - resumes from (M, L, Acc) over K/V rows gathered at selected indices
//   kDense  : plain causal attention (baseline)
//   kRows   : causal attention of any number of query rows over any number of keys (the rows that the sparse operator does
//             not cover: ragged tails, short prompts, prompts continued on a cache), the keys split over work-groups
//   kMasked : the same with a boolean mask (padded batches, sliding windows) instead of the causal rule
//
// Formulation.  A wave owns 32 query rows and computes the TRANSPOSED score tile
//   S^T[key][query] = K[key][:] . Q[query][:]      (MFMA A = K rows from LDS, B = Q from registers)
// so that in the 32x32 accumulator layout a lane holds one query column: the soft-max statistics
// of a query are then plain per-lane scalars (one exchange with the lane 32 positions away
// completes the row max).  The second product is computed transposed as well,
//   O^T[d][query] += V^T[d][key] . P^T[key][query]  (A = V^T, B = P^T straight from the S^T
// accumulator registers, rounded to bf16; rows and masked: as two such numbers) - P never travels through LDS.
// The contraction slot k = 8*(lane/32) + e of MFMA step st of key block kb is fed from accumulator
// register 8*st + e, i.e. key 32*kb + 16*st + 8*(e/4) + 4*(lane/32) + e%4: two runs of four
// consecutive keys.  V sits row-major in LDS exactly as it is in memory, and each run of four keys
// at one head-dim column is fetched with the transposing LDS read ds_read_b64_tr_b16 (within a group
// of 16 lanes, lane i receives column i of the 4x16 block whose rows the group's lanes point at).
//
// A reference m is subtracted inside the first product: the score accumulators start from -m (a per-lane
// constant, kept replicated in a 16-register tuple) instead of zero, so the tile arrives as S - m and
// p = exp2(S - m) needs no subtraction.  m is the running row max: with a probability in one 16-bit number the key that
// weighs most then has p = 1, which is exact (kept at the max of a row's first keys, the error of P.V grows by up to a factor of
// three where few keys weigh much).  Whether a lane's max grew is a comparison of S - m with zero, before the two lanes of
// a row have exchanged anything; only when one did (rare after the first tiles) does the wave take a slow path that completes
// the max, shifts the tile, re-bases the tuple and rescales the accumulators - exact for the lanes whose
// max did not move (shift 0, factor 1).  Where one key outweighs the rest by far, not even the lane's own max is formed (kBySum).  (The exchange on every half-tile instead: 16384 tokens dense, 32/8 heads of 128, 1830 us
// against 1796.)
//
// bf16 rows and masked modes, which keep a probability as two numbers, need no max at all (kLazyRef): m is the row max of the
// first 32 keys and stays, and a larger score gives a p above 1, which is held as precisely as one below.  When the
// sum of a half-tile's p exceeds kRebaseSum - an overflowing exp2 included - the wave forms that half's scores again,
// moves m to the row's max and rescales, before these p are used.  (fp16 forms 2^15 p, which has no room above p = 1.)  What the
// larger p take from the range of V is given back at the end, where sums that overflowed are formed again (aa_nonfinite.h).
// 777 rows over 777 keys, 32/8 heads of 128: 23.0 -> 21.1 us; a padded batch of 3 x 2500: 203 -> 193.
//
// Inside a 64-key tile the two 32-key halves are staggered so that matrix and vector work overlap
// within a wave: S0 | S1 with soft-max(S0) | P0.V0 with soft-max(S1) | P1.V1.  The online soft-max
// therefore advances 32 keys at a time.
//
// Work-group = 4 waves = 128 query rows; keys are consumed 64 at a time through a
// double-buffered LDS tile that the memory system fills directly (global_load_lds_dwordx4: no staging
// registers, no LDS store instructions).  Such a load writes lane L's 16 bytes at M0 + 16*L, so LDS rows
// are unpadded; bank conflicts are avoided by XOR-swizzling the 16-byte chunks of a row, which
// costs nothing on the load side (a lane simply fetches the chunk that belongs in its slot):
//                             head dimension 128                64
//   K row r, chunk c  ->  slot c ^ (r & 15)          c ^ ((r & 7) ^ (r >> 3 & 1))   (row-per-lane 16-byte reads)
//   V row r, chunk c  ->  slot c ^ ((r & 3) << 2)    c ^ ((r & 3) << 1)             (transposing 8-byte reads)
// These choices measure conflict-free for their read pattern: 4 clocks of the LDS a 16-byte read, 2 a transposing one, of which 32 lanes read four
// chunks of four rows at a time, so that those have to lie in sixteen different slots.  (Of 256-byte rows with c ^ ((r & 7) << 1) they lie in eight: 4 clocks;
// 16384 tokens dense, 32/8 heads of 128, LDS busy 4.08e8 -> 2.73e8 clocks, 1735 -> 1730 us.)
#include <cstddef>
#include <type_traits>

#include "aa_common.h"
#include "aa_kernels.h"
#include "aa_nonfinite.h"
#include "aa_threshold.h"

namespace aa {

constexpr int kBN = 64;        // keys per LDS tile
constexpr int kLoadBytes = 4096; // what one LDS-DMA instruction of the work-group brings (256 threads x 16 bytes)
constexpr int kDist = 4;         // MFMA operands are fetched from LDS this many MFMAs ahead of their use
constexpr float kRebaseSum = 16384.f;  // (kLazyRef) largest sum of 16 probabilities that is used as it is
constexpr float kNoRef = -8.5e37f;     // (kLazyRef) reference of a row that has seen no key: what it sees first overflows exp2
constexpr int kIdxWin = 1024;    // selected-key indices held in LDS at a time (16 tiles)
constexpr int32_t kMixedTile = 1 << 30;  // (masked) flag of a listed tile of which some pairs are masked

enum FlashMode : int { kAnchor = 0, kSparse = 1, kDense = 2, kRows = 3, kMasked = 4 };

#ifndef AA_SPARSE_CHAIN
#define AA_SPARSE_CHAIN 1  // 0: every query block of a stage-3 work-group requests its own first tile, queries and state
#endif

typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) shortx4 lds_shortx4;

// Swizzle of the 16-byte chunks of LDS row r (see the top of the file); both have a period of 32 rows or less.
template <int D>
__device__ __forceinline__ int k_swizzle(const int r) { return D == 128 ? r & 15 : (r & 7) ^ ((r >> 3) & 1); }
template <int D>
__device__ __forceinline__ int v_swizzle(const int r) { return D == 128 ? (r & 3) << 2 : (r & 3) << 1; }

template <int MODE, int D, int TEAMS>
struct FlashSmem {
  struct {
    char k[2][kBN * 2 * D];
    char v[2][kBN * 2 * D];
  } t[TEAMS];  // (the epilogue stages the output in the tile space)
  floatx2 stats[TEAMS > 1 ? 256 : 1];  // the second team's reference and sum, lane by lane
  // sparse mode: window of the big block's index list; masked mode: the chunk's tiles that hold a visible key, and their number
  alignas(16) int32_t idx[MODE == kSparse ? kIdxWin : MODE == kMasked ? kMaskedTiles + 4 : 4];
};

// Query pre-scaling into the exp2 domain, eight elements at a time.  `chain`: both constants and both products rounded
// to the tensors' 16-bit type (stage 1, whose definition takes sm_scale as a compile-time constant); otherwise float32
// products and one rounding.
template <typename T>
__device__ __forceinline__ typename T::vec8 scale_q8(const u32x4 raw, const float sm_scale, const bool chain) {
  const uint32_t w[4] = {raw[0], raw[1], raw[2], raw[3]};
  uint32_t o[4];
  if (chain) {  // r16(r16(q * r16(sm_scale)) * r16(log2e))
    const float s16 = T::round(sm_scale), c16 = T::round(kLog2e);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = T::round(T::lo(w[i]) * s16), b = T::round(T::hi(w[i]) * s16);
      o[i] = T::pack(a * c16, b * c16);
    }
  } else {  // float32 products, one rounding
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = T::pack((T::lo(w[i]) * sm_scale) * kLog2e, (T::hi(w[i]) * sm_scale) * kLog2e);
  }
  const u32x4 packed = {o[0], o[1], o[2], o[3]};
  return *reinterpret_cast<const typename T::vec8*>(&packed);
}

// One K/V tile: a row has D/8 slots of 16 bytes and one load instruction of the work-group fills 2048/D rows, thread t slot
// t % (D/8) of row t / (D/8) + (2048/D)*j (j = 0..3 at head dimension 128, 0..1 at 64); tile_fetch_one issues one of the
// tile's eight (four) loads.  `kb`/`vb` are the
// wave-uniform head bases, `k_col`/`v_col` the byte offset of this thread's (swizzled) chunk inside a row,
// `lds_k`/`lds_v` the LDS address of wave w's first slot in the destination tile.  Gathered tiles take their row numbers from
// the LDS window of the index list (a dependent global load per tile would put a full memory latency on the
// critical path of every tile); the caller reads a tile's row numbers (`gather_keys`, see tile_gather_keys)
// before it issues the tile's first load: a wave's LDS reads are served in order with its global -> LDS loads, so a row
// number read after a load would arrive only when that load's data has.
// the row numbers lane `tid` needs for the gathered tile at list position key0 (positions past the count hold 0: row 0,
// masked later)
// (A tile does not cross the window's end: one address, and a lane's rows lie at constant distances from it.  An address each, wrapped: 12
// vector instructions of a tile's 165 more; 32768 tokens with nearly every key selected 8.97 -> 8.91 ms.)
template <int D>
__device__ __forceinline__ void tile_gather_keys(uint32_t (&keys)[D / 32], const int32_t* idx_win, const int key0, const int tid) {
  typedef __attribute__((address_space(3))) uint32_t lds_u32;
  const uint32_t first = lds_addr(idx_win) + 4u * (uint32_t)((key0 & (kIdxWin - 1)) + tid / (D / 8));
#pragma unroll
  for (int j = 0; j < D / 32; ++j) keys[j] = *(const lds_u32*)(uintptr_t)(first + 4u * (uint32_t)((2048 / D) * j));
}

template <int MODE, int D>
__device__ __forceinline__ void tile_fetch_one(const int n, const char* kb, const char* vb, const uint32_t k_row_bytes,
                                               const uint32_t v_row_bytes, const uint32_t k_col, const uint32_t v_col, const int key0,
                                               const uint32_t* gather_keys, const uint32_t lds_k, const uint32_t lds_v,
                                               const uint32_t k_voff, const uint32_t v_voff) {
  constexpr int kLoadRows = 2048 / D;  // rows that one load instruction fills
  const int j = n >> 1;  // load n: K (even n) or V (odd n) rows kLoadRows*j + ...
  if (MODE == kSparse) {
    const uint32_t key = gather_keys[j];  // this lane's row of the tile's j-th block of kLoadRows rows
    if ((n & 1) == 0) load16_to_lds(kb, __umul24(key, k_row_bytes) + k_col, lds_k + j * kLoadBytes);
    else load16_to_lds(vb, __umul24(key, v_row_bytes) + v_col, lds_v + j * kLoadBytes);
  } else if (MODE == kRows || MODE == kMasked) {
    // consecutive keys up to a key count that need not fill the last tile: the caller's per-lane offsets (gather_keys: D/32
    // for K, D/32 for V, from the tile's first row) are loop-invariant except that they are clamped for that tile
    if ((n & 1) == 0) load16_to_lds(kb + (uint64_t)(uint32_t)key0 * k_row_bytes, gather_keys[j], lds_k + j * kLoadBytes);
    else load16_to_lds(vb + (uint64_t)(uint32_t)key0 * v_row_bytes, gather_keys[D / 32 + j], lds_v + j * kLoadBytes);
  } else {
    // consecutive keys: the first row of the tile's j-th block of kLoadRows rows goes into the (scalar) base address, the
    // thread's row inside the block and its chunk are one loop-invariant vector offset - no vector arithmetic per tile
    if ((n & 1) == 0) load16_to_lds(kb + (uint64_t)(uint32_t)(key0 + kLoadRows * j) * k_row_bytes, k_voff, lds_k + j * kLoadBytes);
    else load16_to_lds(vb + (uint64_t)(uint32_t)(key0 + kLoadRows * j) * v_row_bytes, v_voff, lds_v + j * kLoadBytes);
  }
}

// D is the head dimension, 128 or 64: it sets the LDS row pitch, the number of tile loads, of MFMA steps over the head
// dimension (kKS per 32 keys of Q.K^T) and of 32-column output blocks (kDB).
//
// Work-groups per CU: with 128 two (up to 251 registers, 64 KB of LDS).  With 64 a tile has half the MFMAs but the same soft-max, so that the vector
// ALU has more to do than the matrix pipe, and a third wave per SIMD (168 registers; around the tile loop 8 of them spill in sparse mode, 9 in fp16, and 1 in fp16 rows
// mode, alone and beside the anchors) keeps both at work: stage 1 at 16384 tokens, 32/8 heads of 64, fp16, 73 % and 63 % of the cycles, both at once 34 %.  It took 413 us
// instead of 470 with two work-groups per CU and 256-byte LDS rows of which half was filled (371 now).
//
// TEAMS: the waves that own the 128 rows, four to a team.  Two teams take the tiles alternately, each with LDS tiles and accumulators
// of its own, and are merged through LDS at the end, like two chunks of the keys without a launch between them.  This is for
// launches that leave CUs with a single work-group, i.e. one wave to a SIMD, in which the chain scores -> soft-max -> P.V
// of every tile is exposed.  At head dimension 64 a tile of each team takes 2250 to 3000 clocks, two tiles of one team 3100; at 128, where
// the operand reads and tile loads of one team fill more of the LDS's time, 4400 against 3900, so 128 has one team.
template <int MODE, typename T, int D, int TEAMS>
__device__ __forceinline__ void flash_body(const FlashArgs& p, const uint32_t block, FlashSmem<MODE, D, TEAMS>& sm) {
  typedef typename T::vec8 vec8;
  typedef __attribute__((address_space(3))) vec8 lds_vec8;
  typedef FlashSmem<MODE, D, TEAMS> Smem;
  static_assert(offsetof(Smem, idx) % 16 == 0, "the index window is written 16 bytes at a time");
  static_assert(TEAMS == 1 || (TEAMS == 2 && MODE != kSparse && D == 64), "teams");
  constexpr int BM = 128;
  constexpr bool kAnyRows = MODE == kRows || MODE == kMasked;
  constexpr bool kLazyRef = kAnyRows && T::kProbLog2 == 0.f;  // the reference does not follow the row max (see the top of the file)
  // Whether the rounded probabilities are named where they are formed: otherwise the compiler moves half of the exponentials and
  // conversions to the block of their use, where no MFMAs run beside them (131072 tokens, 32/8 heads of 128, all stages: 7.60 ms
  // against 7.53).  Head dimension 64 spills registers for it (anchor, sparse, fp16 rows).
  constexpr bool kPinned = D == 128 || kLazyRef || MODE == kDense;
  // MFMAs of a tile that are issued behind its closing barrier, while the first K operands of the next tile are on their way: with none a wave waits
  // a whole LDS latency there.  0 against 2: dense 16384 tokens, 32/8 heads of 128, 1692.2 -> 1684.7 us, 131072 7080 -> 7040, 32768 with nearly every key selected
  // 8508 -> 8472, rows 777 19.9 -> 19.65, 14/2 heads of 64, 2048 tokens dense 22.1 -> 21.7, 1900 rows 25.5 -> 24.75; three of them, with
  // operands fetched one MFMA before the barrier: 0 to 0.6 % slower than two.  Rows of fp16 at 64 have no registers for the operands: 1493 of 14/2 heads 26.1 -> 28.2,
  // 1700 of 32/8 30.3 -> 34.2; with two teams they have, and 850 to 1000 rows of 32/8 heads are from 1 % slower (no sink) to 2 % faster: none either.
  constexpr int kTail = MODE == kRows && !kLazyRef && D == 64 ? 0 : 2;
  constexpr bool kChecksSums = kLazyRef;
  // What follows a grown max, and the masking of pairs, is laid out of line where it is expected to be rare, which spares what does not follow a jump.  It is
  // not rare where a call is short and no key outweighs the rest: half of the tiles in anchor and dense mode (one time in two against never: dense 1024
  // tokens without a sink, 32/8 heads of 128, 25.3 -> 24.4 us, 2048, 14/2 of 64, fp16 27.4 -> 26.7, with a sink 23.6 -> 22.9; an operator call of one big block,
  // 32/8 of 64, 36.1 -> 35.0; 16384 tokens dense and 131072 of the operator +-0.1 %).  Rows of fp16 at 64 spill out of line, and their maxima grow in the first tiles of
  // every chunk but the first, which holds no sink, and everywhere without one (one time in two, in ten and never: 1493 rows, 14/2 heads, in chunks
  // 25.6, 26.2 and 27.5 us; 1700 rows, 32/8 heads, without a sink 37.2, 37.9 and 41.5, with one 30.3, 29.7 and 30.1).  Lists gain 0.8 % from one in two at
  // 8192 tokens, 14/2 heads of 64, and lose 2 at 4096.  (The masking alone stays out of line in anchor mode: two registers spill for it at 64, 4096 tokens, 14/2
  // heads of 64, few keys selected 73.6 -> 72.9 us, 32/8 106.5 -> 105.9.  In dense mode that gives 0.6 % without a sink and costs 0.6 with one: as the rest.)
  constexpr int kGrows = MODE == kAnchor || MODE == kDense ? 2 : MODE == kRows && !kLazyRef && D == 64 && TEAMS == 1 ? 1 : 0;
  static_assert(D == 128 || D == 64, "head dimension");
  constexpr int kKS = D / 16;       // MFMAs per 32-key block of S^T = K Q^T
  constexpr int kDB = D / 32;       // 32-column blocks of the head dimension: accumulators of O^T
  constexpr int kNS = 2 * kKS;      // S^T slots of a 64-key tile
  constexpr int kNV = 4 * kDB;      // O^T slots of a 64-key tile (two 16-key steps per 32-key block)
  constexpr int kRowBytes = 2 * D;  // pitch of a K/V row in LDS (unpadded, chunks swizzled)
  constexpr int kTileBytes = kBN * kRowBytes;
  constexpr int kSlots = D / 8;              // 16-byte slots of a row
  constexpr int kLoadRows = 256 / kSlots;    // rows that one load instruction of the work-group fills
  constexpr int kHalfLoads = kBN / kLoadRows;  // load instructions of a K (or V) tile

  const int tid = TEAMS > 1 ? threadIdx.x & 255 : threadIdx.x;  // (within the team)
  const int team = TEAMS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  auto& tiles = sm.t[team];
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int c32 = lane & 31;

  // ---- which rows ----------------------------------------------------------------------------
  // A work-group owns 128 query rows - in sparse mode p.q_blocks_per_wg consecutive blocks of 128 rows of one big
  // block, one after the other: they share the big block's index list (fetched once), and the output stores of one
  // block drain while the next one is already loading, instead of every 128 rows paying for a work-group launch, the
  // list's round trip to memory and the wait for its stores.
  const int group = p.group;
  const int nq = MODE == kSparse ? p.q_blocks_per_wg : 1;
  // (anchor, a single big block) The ratio, which a logged call waits for, is known at once.  From the work-group of the first rows, which is dealt out
  // last, it came 5 us later: calls in a row, 2048 tokens, 14/2 heads of 64 28.3 us -> 23.8, 32/8 heads of 64 29.4 -> 27.4.
  if (MODE == kAnchor && p.ratio != nullptr && block == 0 && threadIdx.x == 0) store_ratio(0.f, p.ratio, p.ratio_host);
  // (the sum that stage 2 makes)
  if (MODE == kAnchor && p.clear != nullptr && block == 0 && threadIdx.x == 0) *p.clear = 0;
  // (sparse) one work-group more than the query blocks need, the first, sums the counts to the ratio beside the others
  const bool sums = MODE == kSparse && p.ratio != nullptr;
  if (sums && block == 0) {
    sum_counts(p.counts, p.n_ratio_counts, p.ratio_inverse, p.ratio, p.ratio_host, reinterpret_cast<int64_t*>(sm.idx));
    return;
  }
  const uint32_t wg = block - (sums ? 1u : 0u);
  const int S = p.big_block;
  int g, qunit, bb = 0;
  uint32_t unit, index;  // the KV head, of all batch elements', and the number of the work-group among its
  int chunk = 0;  // (rows) which chunk of the keys
  if (MODE == kSparse && p.pairs) {
    // Stage 3's work per (KV head, big block) pair is the length of the pair's index lists, which depends on the data:
    // a head whose queries select many keys would keep its XCD busy long after the others have finished if whole
    // heads were tied to XCDs.  So the unit that stays on one XCD (and shares its L2) is the pair - the query blocks of
    // a big block and the heads of a KV group gather the same rows - and consecutive pairs, ordered latest big block
    // first, go round-robin over the XCDs with a rotation, so that every XCD sees every head and every depth.
    uint32_t kp = wg / 8u, within = take_remainder(kp, p.by_pair, (uint32_t)(group * p.q_units)), pair = kp * 8u + (wg % 8u + kp) % 8u;
    unit = take_remainder(pair, p.by_units, (uint32_t)p.units);
    bb = p.n_big - 1 - (int)pair;
    g = (int)take_remainder(within, p.by_group, (uint32_t)group);
    qunit = bb * p.q_units + (int)within;
  } else if (kAnyRows) {
    // A work-group owns 128 columns of one KV head - a column is one (query row, head of the group) pair, heads running
    // fastest, so all heads of a group use the same K/V tile - and one chunk of the keys.  Work-groups of one chunk are
    // neighbours on one XCD (they read the same K/V rows), latest columns, which see the most keys, first.
    dealt(p.deal, wg, unit, index);
    qunit = p.n_col_blocks - 1 - (int)take_remainder(index, p.by_cols, (uint32_t)p.n_col_blocks);
    chunk = (int)index;
    g = 0;
  } else {
    dealt(p.deal, wg, unit, index);
    g = (int)take_remainder(index, p.by_group, (uint32_t)group);
    // longest rows first (later big blocks also carry the longest index lists; sparse mode may leave out the first, whose rows select nothing)
    qunit = (MODE == kSparse ? p.n_big * p.q_units : p.n_ctx / BM) - 1 - (int)index;
    // (all blocks of a work-group lie in one big block: the host picks q_blocks_per_wg so)
    if (MODE == kAnchor || MODE == kSparse) bb = (int)quotient((uint32_t)qunit, p.by_block);
  }
  const int b = (int)quotient(unit, p.by_kv_heads), kvh = (int)unit - b * p.n_kv_heads;
  const int hq = kvh * group + g;
  const int64_t bh = (int64_t)b * p.n_q_heads + hq;

  const uint16_t* qp = p.q + b * p.q_sb + hq * p.q_sh;
  const char* kbase = reinterpret_cast<const char*>(p.k + b * p.k_sb + kvh * p.k_sh);
  const char* vbase = reinterpret_cast<const char*>(p.v + b * p.v_sb + kvh * p.v_sh);
  const uint32_t k_row_bytes = (uint32_t)p.k_sn * 2u, v_row_bytes = (uint32_t)p.v_sn * 2u;

  // ---- sparse mode: what the query blocks of a work-group share, and what they hand to each other -------
  // All blocks lie in one big block of one head, so they walk the same index list and gather the same tiles.  When the
  // list fits the LDS window, the blocks are chained: the last tile of a block brings the list's first tile into the idle
  // buffer for the next block, whose queries and statistics are requested before the output of the block is staged and
  // whose accumulator state is requested as soon as the staging has emptied the accumulator registers - so the next
  // block starts its first product without a round trip to memory of its own.
  int cnt = 0, cap = 0, sparse_tiles = 0;
  const int32_t* cbase = nullptr;
  if (MODE == kSparse) {
    cap = max(bb * S - 2 * p.block_size, 0);  // capacity of the big block's list (a multiple of 4)
    // (counts and indices come from device memory the caller filled: a count beyond the capacity or an index beyond
    // the context is clamped rather than followed out of bounds)
    cnt = max(0, min(p.counts[bh * p.n_big + bb], cap));
    cbase = p.coords + bh * p.coords_per_head + coords_tri(bb, S, p.block_size);
    sparse_tiles = (cnt + kBN - 1) / kBN;
  }
  const bool list_chains = MODE == kSparse && AA_SPARSE_CHAIN && sparse_tiles > 0 && sparse_tiles <= kIdxWin / kBN;
  int cur = 0;             // (sparse) LDS buffer of the next tile to be computed
  bool chained = false;    // (sparse) this block's first tile and state were requested by the previous block
  bool have_queries = false;  // (sparse) so were its queries and statistics
  u32x4 qraw[kKS];
  float m_in = 0.f, l_in = 0.f;
  floatx16 acc[kDB];
  // (sparse) queries and soft-max statistics of the block whose lane row is `row`
  auto request_queries = [&](const int row) __attribute__((always_inline)) {
    const uint16_t* qr = qp + (int64_t)row * p.q_sn + 8 * half;
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks) qraw[ks] = *reinterpret_cast<const u32x4*>(qr + 16 * ks);
    m_in = p.M[bh * p.n_ctx + row];
    l_in = half == 0 ? p.L[bh * p.n_ctx + row] : 0.f;  // the two halves are summed at the end
  };
  // (sparse) the accumulator state of that block.  (The accumulator state and the output are touched once each: they
  // are written and read with the non-temporal hint, so that they do not push K/V rows, which many work-groups share,
  // out of the L2.)
  auto request_state = [&](const int row) __attribute__((always_inline)) {
    const float* af = p.acc_frag + ((bh * (p.n_ctx / 32) + row / 32) * (4 * kDB)) * 256 + lane * 4;
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const floatx4 t = __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(af + (db * 4 + rg) * 256));
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[db][rg * 4 + c] = t[c];
      }
  };

  for (int qb = 0; qb < nq; ++qb) {
  const int R0 = (qunit * nq + qb) * BM;
  const int wr0 = R0 + wave * 32;
  // (rows) this lane's column, as (row, head of the group): columns past the last one repeat it and are not stored
  const int n_cols = kAnyRows ? p.n_rows * group : 0;
  const int my_col = min(wr0 + c32, n_cols - 1);
  const int my_row = kAnyRows ? (int)quotient((uint32_t)my_col, p.by_group) : wr0 + c32;
  // (rows) the last key this lane's row sees, and the smallest such key of the wave (rows ascend with the lane)
  const int my_last_key = kAnyRows ? min(p.causal_offset + my_row, p.n_ctx - 1) : my_row;
  const int wave_last_key = kAnyRows ? __builtin_amdgcn_readfirstlane(my_last_key) : wr0;

  // ---- sparse mode: the queries and the softmax statistics are requested first ----------------------
  // They depend on nothing, whereas the first K/V tile needs the index list, which needs its own round trip to
  // memory.  The 64 KB of accumulator state follow the first tile's loads (further down) and are not waited for
  // before the first scores are computed.
  float l_run;
  const uint16_t* qrow = qp + (int64_t)my_row * p.q_sn + 8 * half + (kAnyRows ? (my_col - my_row * group) * p.q_sh : 0);
  if (MODE == kSparse && !have_queries) request_queries(my_row);
  auto load_queries = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks) qraw[ks] = *reinterpret_cast<const u32x4*>(qrow + 16 * ks);
  };
  // Before all else, so that their way from memory is not added to that of the mask's tile flags, on which the first tile waits, or of that tile: masked
  // batches of 300 to 4000 tokens 5 % on average, up to 24 % (3 x 2500, 32/8 heads of 128, 181.4 -> 175.4 us; 2 x 2000, 14/2 of 64, 46.1 -> 39.4; of 96 sizes
  // one 2 % slower and no other more than 1), dense 1024 tokens, 14/2 heads of 64, 14.1 -> 13.85, 777 rows 19.65 -> 19.55, larger
  // launches +-0.2 %.  fp16 rows at 128, which wait longer for the first tile then, 20.3 -> 21.4, and one team's at 64 (1700 of 32/8 heads 30.3 -> 32.1, 1900 of
  // 14/2 27.4 -> 27.8): after it; two teams' 0.7 % faster (930 of 32/8 16.8 -> 16.6).
  constexpr bool kQueriesFirst = MODE != kSparse && (MODE != kRows || kLazyRef || TEAMS == 2);
  if (kQueriesFirst) load_queries();
  const bool feeds_next = list_chains && qb + 1 < nq;  // the next block takes its first tile from this one

  // ---- tile schedule -------------------------------------------------------------------------
  // (anchor) the first big block's rows select no keys further on: where the caller gives the output, they are done here
  const bool finishes = MODE == kAnchor && p.out != nullptr && bb == 0;
  const bool pool = MODE == kAnchor && TEAMS == 1 && p.qbar_out != nullptr && !finishes;  // (two teams: a single big block only)
  int n_tiles, n_init = 0;
  int key_base = 0;  // (rows) first key of the chunk
  int entry_next = 0;  // (masked) list entry of the tile to be fetched next
  int entry_after = 0;  // (masked) and of the one after that, read from LDS a whole tile before it is needed
  u32x2 mask_word_next = {0u, 0u};  // (masked) which of that tile's 64 keys this lane's row sees, if the tile is a mixed one
  const uint32_t mask_row_off = MODE == kMasked ? (uint32_t)my_row * (uint32_t)p.mask_words_per_row * 8u : 0u;  // (below 2^32: checked on the host)
  auto request_mask_word = [&]() __attribute__((always_inline)) {
    if (MODE == kMasked && (entry_next & kMixedTile)) {
      const char* w = reinterpret_cast<const char*>(p.mask_words + ((int64_t)b * p.n_rows * p.mask_words_per_row + (entry_next & (kMixedTile - 1))));
      mask_word_next = *reinterpret_cast<const u32x2*>(w + mask_row_off);
    }
  };
  if (MODE == kAnchor) {
    n_init = min(S, R0 + BM) / kBN;
    n_tiles = n_init + (bb >= 1 ? (R0 + BM - bb * S) / kBN : 0);
  } else if (MODE == kDense) {
    n_tiles = (R0 + BM) / kBN;
  } else if (kAnyRows) {
    const int last_row = min(R0 + BM, n_cols) - 1;
    const int seen = min(p.causal_offset + (int)quotient((uint32_t)last_row, p.by_group), p.n_ctx - 1) / kBN + 1;  // tiles up to the last key any column sees
    key_base = chunk * p.chunk_tiles * kBN;
    n_tiles = min(seen - chunk * p.chunk_tiles, p.chunk_tiles);
    if (n_tiles <= 0) return;  // (never chunk 0: every row sees at least one key)
    if (MODE == kMasked) {
      // list the chunk's tiles in which any row of the work-group sees a key
      if (wave == 0 && team == 0) {
        const uint8_t* flags = p.tile_flags + ((int64_t)b * p.n_col_blocks + qunit) * p.mask_words_per_row + chunk * p.chunk_tiles;
        int listed = 0;
        for (int t = 0; t < n_tiles; t += 64) {
          const int flag = t + lane < n_tiles ? flags[t + lane] : 0;
          const uint64_t some = __ballot(flag != 0);
          if (flag) sm.idx[listed + __popcll(some & ((1ull << lane) - 1))] = (chunk * p.chunk_tiles + t + lane) | (flag == 1 ? kMixedTile : 0);
          listed += __popcll(some);
        }
        if (lane == 0) sm.idx[kMaskedTiles] = listed;
      }
      __syncthreads();
      n_tiles = __builtin_amdgcn_readfirstlane(sm.idx[kMaskedTiles]);
      entry_next = n_tiles > team ? __builtin_amdgcn_readfirstlane(sm.idx[team]) : 0;
      entry_after = sm.idx[max(min(team + TEAMS, n_tiles - 1), 0)];
    }
  } else {
    n_tiles = sparse_tiles;
  }
  // first key (anchor, dense) or first list position (sparse) of tile i
#define AA_TILE_KEY0(i) \
  (MODE == kMasked ? (entry_next & (kMixedTile - 1)) * kBN \
   : (MODE == kAnchor) ? ((i) < n_init ? (i) * kBN : bb * S + ((i) - n_init) * kBN) : (kAnyRows ? key_base : 0) + (i) * kBN)

  // sparse mode: list positions [w0, w0 + kIdxWin) -> LDS (zeros past the count).  The load is bounded by the list's
  // capacity, not by its count, so that it does not have to wait for the count to arrive; what lies past the count is
  // zeroed afterwards.
  auto fill_index_window = [&](const int w0) {
    const int pos = w0 + 4 * tid;
    int4 v = {0, 0, 0, 0};
    if (pos < cap) v = *reinterpret_cast<const int4*>(cbase + pos);  // lists start 16-byte aligned; capacity is a multiple of 4
    if (pos >= cnt) v.x = 0;
    if (pos + 1 >= cnt) v.y = 0;
    if (pos + 2 >= cnt) v.z = 0;
    if (pos + 3 >= cnt) v.w = 0;
    const uint32_t last = (uint32_t)p.n_ctx - 1u;
    v.x = (int)min((uint32_t)v.x, last);
    v.y = (int)min((uint32_t)v.y, last);
    v.z = (int)min((uint32_t)v.z, last);
    v.w = (int)min((uint32_t)v.w, last);
    *reinterpret_cast<int4*>(&sm.idx[4 * tid]) = v;
  };
  // (uniform over the work-group; not conditioned on the count, see above.  Later blocks of the work-group find the
  // list's first window still in place unless the list is longer than the window)
  if (MODE == kSparse && cap > 0 && (qb == 0 || n_tiles > kIdxWin / kBN)) {
    fill_index_window(0);
    __syncthreads();
  }

  // this thread's chunk of a row (swizzled: see the top of the file) and the wave's slice of the LDS tiles
  const uint32_t k_col = (uint32_t)((tid % kSlots) ^ k_swizzle<D>(tid / kSlots)) * 16u;
  const uint32_t v_col = (uint32_t)((tid % kSlots) ^ v_swizzle<D>(tid / kSlots)) * 16u;
  const uint32_t lds_k0 = lds_addr(tiles.k[0]) + wave * 1024, lds_v0 = lds_addr(tiles.v[0]) + wave * 1024;
  // byte offset of this thread's chunk of row tid / kSlots of a block of kLoadRows tile rows from the block's first row
  const uint32_t k_voff = (tid / kSlots) * k_row_bytes + k_col, v_voff = (tid / kSlots) * v_row_bytes + v_col;
  // (anchor mode with pooling) the work-group's raw query rows, fetched like a tile by the last tile's load slots
  const char* qblock = reinterpret_cast<const char*>(qp + (int64_t)R0 * p.q_sn);
  const uint32_t q_row_bytes = (uint32_t)p.q_sn * 2u;
  const uint32_t q_voff = (uint32_t)(tid / kSlots) * q_row_bytes + (uint32_t)(tid % kSlots) * 16u;
  // (rows) per-lane offsets of a tile's blocks of kLoadRows K rows and V rows from the tile's first row, of which
  // `rows_left` lie inside the tensor: lanes past the last key read it again and are masked
  uint32_t row_offs[2 * kHalfLoads];
  // (from an opaque copy of the thread number: the pieces would otherwise occupy registers throughout the tile loop for
  // the one time that the offsets are clamped)
  auto set_row_offs = [&](const int rows_left) __attribute__((always_inline)) {
    int t = tid;
    asm volatile("" : "+v"(t));
    const uint32_t kc = (uint32_t)((t % kSlots) ^ k_swizzle<D>(t / kSlots)) * 16u;
    const uint32_t vc = (uint32_t)((t % kSlots) ^ v_swizzle<D>(t / kSlots)) * 16u;
#pragma unroll
    for (int j = 0; j < kHalfLoads; ++j) {
      const uint32_t r = (uint32_t)min(t / kSlots + kLoadRows * j, rows_left - 1);
      row_offs[j] = __umul24(r, k_row_bytes) + kc;
      row_offs[kHalfLoads + j] = __umul24(r, v_row_bytes) + vc;
    }
  };
  if (kAnyRows) set_row_offs(p.n_ctx - AA_TILE_KEY0(min(team, n_tiles - 1)));
  request_mask_word();
  if (n_tiles > team && !chained) {
    const uint32_t first = MODE == kSparse ? (uint32_t)cur * kTileBytes : 0u;
    uint32_t keys0[kHalfLoads] = {};
    if (MODE == kSparse) tile_gather_keys<D>(keys0, sm.idx, 0, tid);
#pragma unroll
    for (int j = 0; j < 2 * kHalfLoads; ++j)
      tile_fetch_one<MODE, D>(j, kbase, vbase, k_row_bytes, v_row_bytes, k_col, v_col, AA_TILE_KEY0(team), kAnyRows ? row_offs : keys0,
                           lds_k0 + first, lds_v0 + first, k_voff, v_voff);
  }
  // the accumulator state: the youngest loads in flight, first needed by the first P.V product
  if (MODE == kSparse && !chained) request_state(my_row);

  // ---- queries: B operand, pre-scaled into the exp2 domain (rows: as they are, the scores are scaled in float32) -----
  const float score_scale = kAnyRows ? p.sm_scale * kLog2e : 1.f;
  vec8 qreg[kKS];
  {
    const bool chain = (MODE == kAnchor) && (p.scale_mode == 0);
    if (MODE != kSparse && !kQueriesFirst) load_queries();
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks) qreg[ks] = kAnyRows ? *reinterpret_cast<const vec8*>(&qraw[ks]) : scale_q8<T>(qraw[ks], p.sm_scale, chain);
  }

  // ---- running state (sparse mode loaded it at the top) -----------------------------------------
  if (MODE != kSparse) {
    l_run = 0.f;
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
  } else {
    l_run = l_in;
  }

  // m_ref is what the score accumulators are pre-loaded with (negated).  Where it follows the running max, m_over is what S - m_ref
  // has to exceed for a new max: 0, and before the first key of a row (m_ref = 0) -inf.  So m_ref + m_over is the running max
  float m_ref = MODE == kSparse ? m_in : kLazyRef ? kNoRef : 0.f;
  float m_over = MODE == kSparse ? 0.f : -INFINITY;
  floatx16 negm;
#pragma unroll
  for (int r = 0; r < 16; ++r) negm[r] = -m_ref;

  if (MODE == kSparse) {
    // Loads complete in order and the accumulator state was requested last, with 4 * kDB load instructions, so "at most
    // that many outstanding" means: everything requested before it - queries, statistics, tile 0 - has arrived.  The
    // state itself may still be on its way while the first scores are computed (the compiler waits where it is first used).
    // (A chained block has nothing to wait for here: its first tile landed before the previous block's last barrier, and
    // the compiler waits for the queries where they are scaled.  The barrier is still needed - the tile about to be
    // requested lands where the other waves staged their output.)
    if (!chained) {
      if (kDB == 4) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    }
    lds_barrier();  // a barrier that does not wait for the loads still in flight
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // tile 0 has landed in LDS
    __syncthreads();
  }

  // per-lane LDS byte offsets.  K: row c32 (+32*kb), chunk 2*ks + half, swizzled.
  // (absolute LDS addresses into the current buffer; the 32-key half and the row steps are immediate offsets)
  const uint32_t first_buf = MODE == kSparse ? (uint32_t)cur * kTileBytes : 0u;  // (sparse) where this block's first tile lies
  // (sparse: formed per block from an opaque copy of the lane number - hoisted out of the loop over the work-group's
  // blocks, the pieces of these addresses would occupy registers throughout the tile loop)
  int lane_t = lane;
  if (MODE == kSparse) asm volatile("" : "+v"(lane_t));
  const int c32_t = lane_t & 31, half_t = lane_t >> 5;
  uint32_t k_rd[kKS];
#pragma unroll
  for (int ks = 0; ks < kKS; ++ks) k_rd[ks] = lds_addr(tiles.k[0]) + first_buf + c32_t * kRowBytes + (((2 * ks + half_t) ^ k_swizzle<D>(c32_t)) << 4);
  // transposing V read i: a group of 16 lanes covers 16 head-dim columns; lane points at row r0 = 4*half + (lane%16)/4
  // (+ multiples of 8, which the swizzle does not see), bf16 columns 32*(i&3) + 16*((lane>>4)&1) + 4*(lane&3): chunk
  // 4*(i&3) + y0 with y0 < 4, swizzled -> one offset per value of i & 3
  uint32_t v_rd[kDB];
  {
    const int r0 = 4 * half_t + ((lane_t & 15) >> 2);
    const int y0 = 2 * ((lane_t >> 4) & 1) + ((lane_t & 3) >> 1);
#pragma unroll
    for (int m = 0; m < kDB; ++m) v_rd[m] = lds_addr(tiles.v[0]) + first_buf + r0 * kRowBytes + (((4 * m + y0) ^ v_swizzle<D>(r0)) << 4) + 8 * (lane_t & 1);
  }


  // key (or list position) that accumulator register r of 32-key half kb of the tile at key0 stands for
#define AA_KEY_OF(kb, r) (key0 + 32 * (kb) + 8 * ((r) >> 2) + 4 * half + ((r) & 3))
  // causal / list-end mask of one 32-key half (only tiles on the diagonal or at the end of a list need it)
#define AA_RARE(x)                                                                     \
  (kGrows == 2   ? __builtin_expect_with_probability((long)(x), 0, 0.55)              \
   : kGrows == 1 ? __builtin_expect_with_probability((long)(x), 0, 0.9)               \
                 : __builtin_expect(x, 0))
#define AA_MASK(sx, kb)                                                              \
  if (MODE == kMasked) {                                                             \
    if (__builtin_expect(mixed, 0)) {                                                \
      uint32_t seen_ = mask_word[kb];                                                \
      asm volatile("" : "+v"(seen_)); /* (the bits are taken apart here, not earlier) */ \
      _Pragma("unroll") for (int r = 0; r < 16; ++r)                                 \
        if (!((seen_ >> (8 * (r >> 2) + (r & 3))) & 1u)) sx[r] = -INFINITY;          \
    }                                                                                \
  } else if (MODE != kSparse) {                                                      \
    if (MODE == kAnchor ? __builtin_expect(key0 + 32 * (kb) + 31 > wave_last_key, 0) : AA_RARE(key0 + 32 * (kb) + 31 > wave_last_key)) { \
      _Pragma("unroll") for (int r = 0; r < 16; ++r)                                 \
        if (AA_KEY_OF(kb, r) > my_last_key) sx[r] = -INFINITY;                       \
    }                                                                                \
  } else if (__builtin_expect(key0 + 32 * (kb) + 32 > cnt, 0)) {                     \
    _Pragma("unroll") for (int r = 0; r < 16; ++r)                                   \
      if (AA_KEY_OF(kb, r) >= cnt) sx[r] = -INFINITY;                                \
  }
  // this lane's max of one half (the lane 32 positions away holds the other keys of the same query)
#define AA_LANEMAX(sx, mx)                                                           \
  {                                                                                  \
    float t0 = fmaxf(fmaxf(sx[0], sx[1]), sx[2]), t1 = fmaxf(fmaxf(sx[3], sx[4]), sx[5]);      \
    float t2 = fmaxf(fmaxf(sx[6], sx[7]), sx[8]), t3 = fmaxf(fmaxf(sx[9], sx[10]), sx[11]);    \
    float t4 = fmaxf(fmaxf(sx[12], sx[13]), sx[14]);                                 \
    t0 = fmaxf(fmaxf(t0, t1), t2);                                                   \
    t3 = fmaxf(fmaxf(t3, t4), sx[15]);                                               \
    mx = fmaxf(t0, t3);                                                              \
  }
  // (rows: maxima and scores are kept as raw dot products; the scale is applied to the difference, in float32)
#define AA_EXP2(x) fast_exp2(kAnyRows ? (x) * score_scale : (x))
#define AA_PROB(x) (kAnyRows ? prob_exp2<T>(x, score_scale) : AA_EXP2(x))
  // p = exp2(s) (rows: 2^kProbLog2 times that) for accumulator registers 4c .. 4c+3 of one half, summed and rounded into the P^T fragment words
#define AA_EXP_CHUNK(sx, pw, sum, c)                                                 \
  {                                                                                  \
    const float e0 = AA_PROB(sx[4 * (c) + 0]), e1 = AA_PROB(sx[4 * (c) + 1]);        \
    const float e2 = AA_PROB(sx[4 * (c) + 2]), e3 = AA_PROB(sx[4 * (c) + 3]);        \
    sum += e0; sum += e1; sum += e2; sum += e3;                                        \
    pw[(c) >> 1][2 * ((c) & 1) + 0] = T::pack(e0, e1);                                 \
    pw[(c) >> 1][2 * ((c) & 1) + 1] = T::pack(e2, e3);                                 \
    if (kPinned) asm volatile("" : "+v"(pw[(c) >> 1][2 * ((c) & 1) + 0]), "+v"(pw[(c) >> 1][2 * ((c) & 1) + 1]));   \
    if (kAnyRows) { /* what the rounding left, as a second 16-bit number */            \
      pw##_rest[(c) >> 1][2 * ((c) & 1) + 0] = T::pack_rest(e0, e1, pw[(c) >> 1][2 * ((c) & 1) + 0]);  \
      pw##_rest[(c) >> 1][2 * ((c) & 1) + 1] = T::pack_rest(e2, e3, pw[(c) >> 1][2 * ((c) & 1) + 1]);  \
    }                                                                                  \
  }
  // V operand fetch i (two transposing reads): i = (kb*2 + st)*kDB + db
#define AA_V_SRC(i) (v_rd[(i) % kDB] + (uint32_t)(rd_off + (32 * ((i) / (2 * kDB)) + 16 * (((i) / kDB) & 1)) * kRowBytes))
#define AA_V_FETCH(i)                                                                                  \
  {                                                                                                    \
    vlo[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(uintptr_t)(AA_V_SRC(i)));                     \
    vhi[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(uintptr_t)(AA_V_SRC(i) + 8u * kRowBytes));    \
  }
#define AA_PV_MFMA(i, pw)                                                                              \
  {                                                                                                    \
    typedef short shortx8 __attribute__((ext_vector_type(8)));                                         \
    const shortx8 av = __builtin_shufflevector(vlo[i], vhi[i], 0, 1, 2, 3, 4, 5, 6, 7);                \
    acc[(i) % kDB] = T::mfma(*reinterpret_cast<const vec8*>(&av),                                      \
                             *reinterpret_cast<const vec8*>(&pw[((i) / kDB) & 1]), acc[(i) % kDB]); \
    if (kAnyRows) acc[(i) % kDB] = T::mfma(*reinterpret_cast<const vec8*>(&av),                        \
                                           *reinterpret_cast<const vec8*>(&pw##_rest[((i) / kDB) & 1]), acc[(i) % kDB]); \
  }
#define AA_FENCE __builtin_amdgcn_sched_barrier(0)
  // scores of 32-key half kb of the tile whose K rows lie at immediate offset rd, from c_init on
#define AA_SCORES(sx, kb, rd, c_init)                                                                                   \
  _Pragma("unroll") for (int ks = 0; ks < kKS; ++ks)                                                                    \
    sx = T::mfma(*(const lds_vec8*)(uintptr_t)(k_rd[ks] + (uint32_t)((rd) + 32 * (kb) * kRowBytes)), qreg[ks], ks == 0 ? c_init : sx);
  const floatx16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  if (kLazyRef && n_tiles > team) {  // the reference: the row max of the first 32 keys
    const int key0 = AA_TILE_KEY0(team);
    const bool mixed = MODE == kMasked && (entry_next & kMixedTile);
    const u32x2 mask_word = {mask_word_next[0] >> (4 * half), mask_word_next[1] >> (4 * half)};
    floatx16 sx;
    float mx;
    AA_SCORES(sx, 0, 0, zero16)
    AA_MASK(sx, 0)
    AA_LANEMAX(sx, mx)
    mx = max_with_other_half(mx);
    m_ref = mx == -INFINITY ? kNoRef : mx;
#pragma unroll
    for (int r = 0; r < 16; ++r) negm[r] = -m_ref;
  }

  // Where the reference follows the running max, a key above it has a probability of 1 or more, so a lane whose 16 probabilities of a
  // half-tile sum to less has none: once a wave's sums have been low (an attention sink: the rest of the keys weigh little), tiles
  // without masked pairs are run without forming maxima (kFew) until a sum says otherwise.  (Compared as bits: a NaN counts as large.  The limit is 1
  // less what rounding can take from a sum; sums have to be half of it to begin, so that ones about it do not end at once what they began: 0.25 or 0.75
  // there cost 0.3 to 0.6 % at sinks 6 nats above the rest, and change the others by less than 0.3.)
  // These tiles have loops of their own: a choice inside a tile costs the branches and register copies that it saves maxima.  131072 tokens,
  // 32/8 heads of 128, few keys selected 7.71 -> 7.44 ms; 16384 dense 1875 -> 1810 us; 16384 fp16, heads of 64, 472 -> 451.  Without a sink nothing is gained.
  //
  // A tile in such a loop saves a twentieth of a tile, and leaving it costs a fourth (the half-tile's scores and exponentials once more, and the way into the
  // other loops).  So a wave leaves twice for nothing, and then once for every kLeaving tiles that it has run.  8192 tokens dense, 32/8 heads of 128, maxima in all
  // tiles, re-entered at once and with 48 tiles to pay (16, 32): a sink 9 nats above the rest 468 us, 450 and 450; 0.1 % of the keys as strong 478, 475, 474; 0.5 %
  // 486, 496, 486 (489, 486); 2 % 512, 532, 515 (518, 514); a new maximum every 250 keys 483, 502, 482; every 33 574, 570, 571.  54 such inputs of both head
  // dimensions: from 4.7 % faster to 0.7 % slower than with all maxima, 0.7 % faster on average; re-entered at once 17 were slower, by up to 5 %.
  constexpr bool kBySum = !kAnyRows;
  constexpr int kLeaving = 48 * TEAMS;
  const uint32_t kSumLimit = __float_as_uint(0.999f), kSumLow = __float_as_uint(0.5f);
  bool few = false;
  int paid_until = -kLeaving;    // the tile from which the next leaving is paid for
  int few_from = 0x7fffffff;     // ... if the last tile's sums were low, the tile from which these loops may be entered

  // One tile.  The LDS buffer it reads (BUF) is a compile-time constant - the loops below are unrolled by two - so that
  // the buffer's offset is part of every LDS instruction's immediate offset and the read addresses are loop-invariant.
  // Sparse mode, whose tile counts can be odd, keeps one copy of each kind of tile (BUF = -1): the buffer is i & 1 and the read
  // addresses step back and forth between the two buffers.  So does masked mode, for which two copies spill 25 registers.
  int32_t buf_step = (MODE == kSparse && cur) ? -kTileBytes : kTileBytes;
  vec8 k_first[kDist];  // the K operands of the next tile's first slots
  if (kTail > 0 && n_tiles > team) {
#pragma unroll
    for (int t = 0; t < kDist; ++t) k_first[t] = *(const lds_vec8*)(uintptr_t)(k_rd[t % kKS] + 32 * (t / kKS) * kRowBytes);
  }
  auto tile = [&](auto buf_const, auto few_const, const int i) __attribute__((always_inline)) {
    constexpr int kBuf = decltype(buf_const)::value;
    constexpr bool kFew = decltype(few_const)::value;
    constexpr uint32_t rd_off = kBuf > 0 ? kBuf * kTileBytes : 0;  // immediate part of the LDS read addresses
    const int buf = kBuf >= 0 ? kBuf : cur;
    const int key0 = AA_TILE_KEY0(i);  // (masked: entry_next is still this tile's)
    const bool mixed = MODE == kMasked && (entry_next & kMixedTile);
    const u32x2 mask_word = {mask_word_next[0] >> (4 * half), mask_word_next[1] >> (4 * half)};
    if (MODE == kSparse && i + 1 < n_tiles && ((i + 1) & (kIdxWin / kBN - 1)) == 0) {
      // tile i+1 opens the next window; everyone finished reading the old one before the last barrier
      fill_index_window((i + 1) * kBN);
      __syncthreads();
    }
    // Tile i+1 goes straight into the other buffer (every wave finished reading it before the last barrier).  Its
    // eight load instructions are spread over the first MFMAs of this tile: issued in one burst by all four waves
    // they queue up behind each other in the memory pipeline and every wave stalls for the length of the queue.
    // (the last tile fetches itself once more into the idle buffer, which keeps the instruction stream free of branches -
    // unless the work-group also pools its queries: then the eight load slots of the last tile bring the work-group's
    // 128 raw query rows into the idle buffer instead, rows 0..63 where K tiles go and rows 64..127 where V tiles go,
    // chunks in place)
    // (sparse, chained: the last tile of a block fetches the list's first tile, for the next block)
    const int i_next = i + TEAMS < n_tiles ? i + TEAMS : (feeds_next ? 0 : i);
    if (MODE == kMasked) {
      entry_next = __builtin_amdgcn_readfirstlane(entry_after);
      request_mask_word();
      entry_after = sm.idx[min(i + 2 * TEAMS, n_tiles - 1)];
    }
    const int key0_next = AA_TILE_KEY0(i_next);
    const bool fetch_queries = MODE == kAnchor && !kFew && pool && i + 1 == n_tiles;  // wave-uniform (a window's last tile has masked pairs)
    // (selects, not branches: the eight slots stay straight-line code; the base address is scalar, and the vector offset
    // is chosen once per tile and operand kind)
    const uint32_t k_voff_sel = fetch_queries ? q_voff : k_voff, v_voff_sel = fetch_queries ? q_voff : v_voff;
    uint32_t keys_next[kHalfLoads] = {};  // (sparse) row numbers of the next tile, read before the tile's first load is issued
    if (MODE == kSparse) tile_gather_keys<D>(keys_next, sm.idx, key0_next, tid);
    if (kAnyRows && p.n_ctx - key0_next < kBN) set_row_offs(p.n_ctx - key0_next);
#define AA_FETCH_ONE(n)                                                                                               \
  if (MODE == kAnchor) {                                                                                              \
    const int j_ = (n) >> 1;                                                                                          \
    const char* kv_ = ((n) & 1) ? vbase + (uint64_t)(uint32_t)(key0_next + kLoadRows * j_) * v_row_bytes                     \
                                : kbase + (uint64_t)(uint32_t)(key0_next + kLoadRows * j_) * k_row_bytes;                    \
    const char* q_ = qblock + (uint64_t)(64 * ((n) & 1) + kLoadRows * j_) * q_row_bytes;                                     \
    load16_to_lds(fetch_queries ? q_ : kv_, ((n) & 1) ? v_voff_sel : k_voff_sel,                                      \
                  (((n) & 1) ? lds_v0 : lds_k0) + (buf ^ 1) * kTileBytes + j_ * kLoadBytes);                      \
  } else {                                                                                                            \
    tile_fetch_one<MODE, D>(n, kbase, vbase, k_row_bytes, v_row_bytes, k_col, v_col, key0_next,                          \
                         kAnyRows ? row_offs : keys_next, lds_k0 + (buf ^ 1) * kTileBytes, lds_v0 + (buf ^ 1) * kTileBytes, k_voff, v_voff);           \
  }
    // (a wave whose rows all lie above this tile - two of the four waves on the last tile of a causal work-group -
    // runs it fully masked: it would only wait at the barrier for the others anyway)
    {
      floatx16 s0, s1;
      vec8 ka[kNS];                // K operand of slot n = kb*kKS + ks
      shortx4 vlo[kNV], vhi[kNV];  // V operand of slot kNS + i, i = (kb*2 + st)*kDB + db
      u32x4 pw0[2], pw1[2];        // P^T fragments (bf16 pairs) of the two halves
      u32x4 pw0_rest[2], pw1_rest[2];  // (rows) and of what their rounding left
      float sum0 = 0.f, sum1 = 0.f;
      float mx0, mx1, shift0 = 0.f, alpha1 = 1.f;  // (where the reference follows the running max)
      bool moved0 = false, moved1 = false;
      // The half whose probabilities sum to more than kRebaseSum once more, from a reference that is the row's max.  (Its
      // scores start from zero: those of a row that had no reference hold nothing but kNoRef.)
      auto rebase = [&](auto kb_const, floatx16& sx, u32x4 (&pw)[2], u32x4 (&pw_rest)[2], float& sum) __attribute__((always_inline)) {
        constexpr int kb = decltype(kb_const)::value;
        float mx;
        AA_SCORES(sx, kb, rd_off, zero16)
        AA_MASK(sx, kb)
        AA_LANEMAX(sx, mx)
        const float m_new = fmaxf(m_ref, max_with_other_half(mx));
        const float alpha = AA_EXP2(m_ref - m_new);
        m_ref = m_new;
        l_run *= alpha;
#pragma unroll
        for (int r = 0; r < 16; ++r) sx[r] -= m_new;
#pragma unroll
        for (int r = 0; r < 16; ++r) negm[r] = -m_new;
#pragma unroll
        for (int db = 0; db < kDB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
        sum = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) { AA_EXP_CHUNK(sx, pw, sum, c) }
      };
      (void)rebase;
      // (kFew) A half whose probabilities do not sum to less than 1 once more, the row's max looked at, as a tile without kFew does: the same bits.
      auto look_again = [&](auto kb_const, floatx16& sx, u32x4 (&pw)[2], u32x4 (&pw_rest)[2], float& sum) __attribute__((always_inline)) {
        constexpr int kb = decltype(kb_const)::value;
        float mx;
        AA_SCORES(sx, kb, rd_off, negm)
        AA_LANEMAX(sx, mx)
        if (__any(mx > m_over)) {
          const float m_new = fmaxf(m_ref + m_over, m_ref + max_with_other_half(mx));
          const float m_base = m_new == -INFINITY ? 0.f : m_new;
          const float alpha = AA_EXP2(m_ref + m_over - m_base), shift = m_base - m_ref;
          m_ref = m_base;
          l_run *= alpha;
#pragma unroll
          for (int r = 0; r < 16; ++r) sx[r] -= shift;
          if (kb == 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s1[r] -= shift;
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) negm[r] = -m_base;
#pragma unroll
          for (int db = 0; db < kDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
        }
        sum = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) { AA_EXP_CHUNK(sx, pw, sum, c) }
        few = false;
        paid_until += kLeaving;
      };
      (void)look_again;
#define AA_K_FETCH(t) ka[t] = *(const lds_vec8*)(uintptr_t)(k_rd[(t) % kKS] + (uint32_t)(rd_off + 32 * ((t) / kKS) * kRowBytes))

      // The MFMAs of a tile are slots 0 .. kNS + kNV - 1 (head dimension 128: 16 for S^T, then 16 for O^T); the operand of
      // slot n is fetched from LDS while slot n - kDist is issued.  The scheduling fences keep that distance: left
      // alone, the reads sink next to their use and every MFMA then waits out a full LDS latency.
#define AA_OPERAND_FETCH(n)                          \
  {                                                  \
    if ((n) < kNS) {                                 \
      AA_K_FETCH((n) % kNS);                         \
    } else if ((n) < kNS + kNV) {                    \
      AA_V_FETCH(((n) - kNS) % kNV)                  \
    }                                                \
  }
#define AA_S_MFMA(sx, n) sx = T::mfma(ka[n], qreg[(n) % kKS], ((n) % kKS) == 0 ? negm : sx)
      // Each half-tile product is kKS (S^T) or 2*kDB (O^T) MFMAs long; the soft-max of the other half sits between them:
      // a quarter of the MFMAs, the row max, half of the MFMAs with the four exp chunks spread over them, the last quarter.
      constexpr int kSPre = kKS / 4, kSMid = kKS / 2, kVPre = kDB / 2, kVMid = kDB;
#pragma unroll
      for (int n = 0; n < kDist; ++n) {
        if (kTail > 0) ka[n] = k_first[n];
        else AA_OPERAND_FETCH(n)
      }
      AA_FENCE;

      // ---- phase A: S0^T = K0 Q^T (and the next tile's eight loads) -------------------------------
#pragma unroll
      for (int n = 0; n < kKS; ++n) {
        AA_OPERAND_FETCH(n + kDist)
        AA_S_MFMA(s0, n);
#pragma unroll
        for (int u = 0; u < 2 * kHalfLoads / kKS; ++u) { AA_FETCH_ONE(n * (2 * kHalfLoads / kKS) + u) }
        AA_FENCE;
      }

      // ---- phase B: S1^T = K1 Q^T, with the soft-max of S0 between the MFMAs ---------------------
#pragma unroll
      for (int n = kKS; n < kKS + kSPre; ++n) {
        AA_OPERAND_FETCH(n + kDist)
        AA_S_MFMA(s1, n);
        AA_FENCE;
      }
      if (!kFew) { AA_MASK(s0, 0) }
      if (!kLazyRef && !kFew) {
        AA_LANEMAX(s0, mx0)
        moved0 = __any(mx0 > m_over);
        if (AA_RARE(moved0)) {
          // some row's max grew.  Lanes whose max did not move get shift 0 and alpha 1 (exact).
          // S1 is being accumulated on top of the old -m_ref and is shifted once it is complete.
          // (a chunk may hold no key of a row's so far - its max stays -inf and its reference 0)
          const float m_new = fmaxf(m_ref + m_over, m_ref + max_with_other_half(mx0));
          const float m_base = m_new == -INFINITY ? 0.f : m_new;
          const float alpha = AA_EXP2(m_ref + m_over - m_base);
          shift0 = m_base - m_ref;
          m_ref = m_base;
          if (MODE != kSparse) m_over = m_new == -INFINITY ? -INFINITY : 0.f;
          l_run *= alpha;
#pragma unroll
          for (int r = 0; r < 16; ++r) s0[r] -= shift0;
#pragma unroll
          for (int r = 0; r < 16; ++r) negm[r] = -m_base;
#pragma unroll
          for (int db = 0; db < kDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
        }
      }
      AA_FENCE;
#pragma unroll
      for (int n = kKS + kSPre; n < kKS + kSPre + kSMid; ++n) {
        AA_OPERAND_FETCH(n + kDist)
        AA_S_MFMA(s1, n);
#pragma unroll
        for (int u = 0; u < 4 / kSMid; ++u) { AA_EXP_CHUNK(s0, pw0, sum0, (n - kKS - kSPre) * (4 / kSMid) + u) }
        AA_FENCE;
      }
#pragma unroll
      for (int n = kKS + kSPre + kSMid; n < kNS; ++n) {
        AA_OPERAND_FETCH(n + kDist)
        AA_S_MFMA(s1, n);
        AA_FENCE;
      }
      if (kChecksSums && __builtin_expect(__any(sum0 > kRebaseSum), 0)) {
        rebase(std::integral_constant<int, 0>{}, s0, pw0, pw0_rest, sum0);
        AA_SCORES(s1, 1, rd_off, negm)
      }
      if (kFew && __builtin_expect(__any(__float_as_uint(sum0) >= kSumLimit), 0)) look_again(std::integral_constant<int, 0>{}, s0, pw0, pw0_rest, sum0);
      l_run += sum0;

      // ---- phase C: O^T += V0^T P0^T, with the soft-max of S1 between the MFMAs --------------------
#pragma unroll
      for (int n = kNS; n < kNS + kVPre; ++n) {
        AA_OPERAND_FETCH(n + kDist)
        AA_PV_MFMA(n - kNS, pw0)
        AA_FENCE;
      }
      if (!kLazyRef && !kFew && AA_RARE(moved0)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s1[r] -= shift0;
      }
      if (!kFew) { AA_MASK(s1, 1) }
      if (!kLazyRef && !kFew) {
        AA_LANEMAX(s1, mx1)
        moved1 = __any(mx1 > m_over);
        if (AA_RARE(moved1)) {
          // as above, except that O^T is rescaled only after the P0 V0 products in flight have been added
          const float m_new = fmaxf(m_ref + m_over, m_ref + max_with_other_half(mx1));
          const float m_base = m_new == -INFINITY ? 0.f : m_new;
          alpha1 = AA_EXP2(m_ref + m_over - m_base);
          const float shift = m_base - m_ref;
          m_ref = m_base;
          if (MODE != kSparse) m_over = m_new == -INFINITY ? -INFINITY : 0.f;
          l_run *= alpha1;
#pragma unroll
          for (int r = 0; r < 16; ++r) s1[r] -= shift;
#pragma unroll
          for (int r = 0; r < 16; ++r) negm[r] = -m_base;
        }
      }
      AA_FENCE;
#pragma unroll
      for (int n = kNS + kVPre; n < kNS + kVPre + kVMid; ++n) {
        AA_OPERAND_FETCH(n + kDist)
        AA_PV_MFMA(n - kNS, pw0)
#pragma unroll
        for (int u = 0; u < 4 / kVMid; ++u) { AA_EXP_CHUNK(s1, pw1, sum1, (n - kNS - kVPre) * (4 / kVMid) + u) }
        AA_FENCE;
      }
#pragma unroll
      for (int n = kNS + kVPre + kVMid; n < kNS + 2 * kDB; ++n) {
        AA_OPERAND_FETCH(n + kDist)
        AA_PV_MFMA(n - kNS, pw0)
        AA_FENCE;
      }
      if (!kLazyRef && !kFew && AA_RARE(moved1)) {
#pragma unroll
        for (int db = 0; db < kDB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[db][r] *= alpha1;
      }
      if (kChecksSums && __builtin_expect(__any(sum1 > kRebaseSum), 0)) rebase(std::integral_constant<int, 1>{}, s1, pw1, pw1_rest, sum1);
      if (kFew) {
        if (__builtin_expect(__any(__float_as_uint(sum1) >= kSumLimit), 0)) look_again(std::integral_constant<int, 1>{}, s1, pw1, pw1_rest, sum1);
      } else if (kBySum) {
        few_from = __any(max(max(__float_as_uint(sum0), __float_as_uint(sum1)), __float_as_uint(m_over)) >= kSumLow) ? 0x7fffffff : paid_until;
      }
      l_run += sum1;

      // ---- phase D: O^T += V1^T P1^T, and the hand-over to the next tile ----------------------------
#pragma unroll
      for (int n = kNS + 2 * kDB; n < kNS + kNV - kTail; ++n) {
        AA_OPERAND_FETCH(n + kDist)
        AA_PV_MFMA(n - kNS, pw1)
        AA_FENCE;
      }
      if (kBuf < 0) {  // the read addresses follow the tiles into the other buffer
#pragma unroll
        for (int ks = 0; ks < kKS; ++ks) k_rd[ks] += buf_step;
#pragma unroll
        for (int m = 0; m < kDB; ++m) v_rd[m] += buf_step;
        buf_step = -buf_step;
        cur ^= 1;
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's share of tile i+1 has landed in LDS
      // (so has the mask word: named here, or the compiler would wait for it behind the next tile's loads)
      if (MODE == kMasked) asm volatile("" : "+v"(mask_word_next[0]), "+v"(mask_word_next[1]));
      __syncthreads();
      AA_FENCE;
      constexpr uint32_t rd_next = kBuf == 0 ? kTileBytes : 0;
#pragma unroll
      for (int t = 0; t < (kTail > 0 ? kDist : 0); ++t) k_first[t] = *(const lds_vec8*)(uintptr_t)(k_rd[t % kKS] + (uint32_t)(rd_next + 32 * (t / kKS) * kRowBytes));
      AA_FENCE;
#pragma unroll
      for (int n = kNS + kNV - kTail; n < kNS + kNV; ++n) {
        AA_PV_MFMA(n - kNS, pw1)
        AA_FENCE;
      }
#undef AA_OPERAND_FETCH
#undef AA_S_MFMA
#undef AA_K_FETCH
    }
#undef AA_FETCH_ONE

  };
  // (a tile without masked pairs, by its number)
  auto whole = [&](const int i) __attribute__((always_inline)) {
    const int key0 = AA_TILE_KEY0(i);
    return MODE == kSparse ? key0 + kBN <= cnt : key0 + kBN - 1 <= wave_last_key;
  };
  typedef std::integral_constant<int, 0> Buf0;
  typedef std::integral_constant<int, 1> Buf1;
  typedef std::integral_constant<int, -1> BufCur;
  int i = team;
  while (i < n_tiles) {
    if (MODE == kSparse || MODE == kMasked) {
      do {
        tile(BufCur{}, std::false_type{}, i);
        i += TEAMS;
      } while (i < n_tiles && !(kBySum && i >= few_from && whole(i)));
      if constexpr (kBySum) {
        few = true;
        while (i < n_tiles && few && whole(i)) {
          tile(BufCur{}, std::true_type{}, i);
          i += TEAMS;
        }
      }
    } else {
      // (anchor, dense: 128 query rows and 64-key tiles, so the window of a query block holds an even number of tiles)
      do {
        tile(Buf0{}, std::false_type{}, i);
        if ((kAnyRows || TEAMS > 1) && i + TEAMS >= n_tiles) { i += TEAMS; break; }
        tile(Buf1{}, std::false_type{}, i + TEAMS);
        i += 2 * TEAMS;
      } while (i < n_tiles && !(kBySum && i >= few_from && i + TEAMS < n_tiles && whole(i + TEAMS)));
      if constexpr (kBySum) {
        few = true;
        while (i + TEAMS < n_tiles && few && whole(i + TEAMS)) {
          tile(Buf0{}, std::true_type{}, i);
          tile(Buf1{}, std::true_type{}, i + TEAMS);
          i += 2 * TEAMS;
        }
      }
    }
  }
  if (TEAMS > 1 && team == 1 && n_tiles % TEAMS != 0) __syncthreads();  // (the barrier of the first team's last tile)
#undef AA_TILE_KEY0
#undef AA_KEY_OF
#undef AA_MASK
#undef AA_RARE
#undef AA_LANEMAX
#undef AA_PROB
#undef AA_EXP_CHUNK
#undef AA_V_SRC
#undef AA_V_FETCH
#undef AA_PV_MFMA
#undef AA_FENCE
#undef AA_SCORES

  const float acc_sum = kAnyRows ? sum_of_all(acc) : 0.f;
  if (kAnyRows && __builtin_expect(__any((kLazyRef ? !is_finite(acc_sum) : is_nan(acc_sum)) && !is_nan(l_run)), 0)) {
    // V holds infinities or NaN, or is too large for probabilities above 1: the wave's sums once more (see aa_nonfinite.h)
    auto each_half = [&](auto&& visit) __attribute__((always_inline)) {
      for (int i = 0; i < 2 * n_tiles; ++i) {  // 32 keys at a time
        if (TEAMS > 1 && (i >> 1) % TEAMS != team) continue;
        int key0 = key_base + 32 * i;
        uint32_t seen;
        if (MODE == kMasked) {
          const int32_t entry = __builtin_amdgcn_readfirstlane(sm.idx[i >> 1]);
          const int tile = entry & (kMixedTile - 1);
          key0 = tile * kBN + 32 * (i & 1);
          seen = ~0u;
          if (entry & kMixedTile) {
            const char* w = reinterpret_cast<const char*>(p.mask_words + ((int64_t)b * p.n_rows * p.mask_words_per_row + tile));
            seen = *reinterpret_cast<const uint32_t*>(w + mask_row_off + 4 * (i & 1));
          }
        } else {
          const int count = my_last_key + 1 - key0;
          seen = count >= 32 ? ~0u : count <= 0 ? 0u : (1u << count) - 1u;
        }
        visit(key0, seen);
      }
    };
    if (kLazyRef) {
      float mx = -INFINITY;
      each_half([&](const int key0, const uint32_t seen) __attribute__((always_inline)) {
        mx = exact_max(exact_scores<T, D>(qreg, kbase, k_row_bytes, key0, p.n_ctx, lane), seen, lane, mx);
      });
      mx = max_with_other_half(mx);
      if (m_ref != kNoRef) {
        l_run *= AA_EXP2(m_ref - mx);
        m_ref = mx;
      }
    }
    const float m_base = m_ref == kNoRef ? 0.f : m_ref;
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
    each_half([&](const int key0, const uint32_t seen) __attribute__((always_inline)) {
      exact_pv_tile<T, D>(acc, qreg, kbase, vbase, k_row_bytes, v_row_bytes, key0, p.n_ctx, seen, m_base, score_scale, lane);
    });
  }

  if (TEAMS > 1) {
    // ---- the second team's state -> the first ----------------------------------------------------
    char* state = sm.t[1].k[0];  // (its tiles: as many bytes as its accumulators)
    static_assert(sizeof(sm.t[0]) == 256 * D / 2 * sizeof(float), "a team's accumulators fill its tile space");
    const float m_own = !kLazyRef ? m_ref + m_over : m_ref == kNoRef ? -INFINITY : m_ref;
    if (team == 1) {
#pragma unroll
      for (int db = 0; db < kDB; ++db)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          floatx4 t;
#pragma unroll
          for (int c = 0; c < 4; ++c) t[c] = acc[db][rg * 4 + c];
          *reinterpret_cast<floatx4*>(state + (db * 4 + rg) * 4096 + tid * 16) = t;
        }
      sm.stats[tid] = floatx2{m_own, l_run};
    }
    __syncthreads();
    if (team == 1) return;  // (barriers further down count the waves that are left)
    const floatx2 other = sm.stats[tid];
    const float m_new = fmaxf(m_own, other[0]), m_base = m_new == -INFINITY ? 0.f : m_new;
    // (bf16 rows: half of both, sums and state alike, so that two finite parts have a finite sum; all chunks have this factor)
    constexpr float kShare = kLazyRef ? 0.5f : 1.f;
    const float w_own = AA_EXP2(m_own - m_base) * kShare, w_other = AA_EXP2(other[0] - m_base) * kShare;
    l_run = l_run * w_own + other[1] * w_other;
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const floatx4 t = *reinterpret_cast<const floatx4*>(state + (db * 4 + rg) * 4096 + tid * 16);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[db][rg * 4 + c] = acc[db][rg * 4 + c] * w_own + t[c] * w_other;
      }
    m_ref = kLazyRef && m_new == -INFINITY ? kNoRef : m_base;
    if (m_new != -INFINITY) m_over = 0.f;
  }
#undef AA_EXP2

  // ---- epilogue --------------------------------------------------------------------------------
  const float l_tot = l_run + xor32(l_run);
  const float m_run = !kLazyRef ? m_ref + m_over : m_ref == kNoRef ? -INFINITY : m_ref;
  if (MODE == kAnchor && !finishes) {
    if (half == 0) {
      p.M_out[bh * p.n_ctx + my_row] = m_run;
      p.L_out[bh * p.n_ctx + my_row] = l_tot;
    }
    float* af = p.acc_out + ((bh * (p.n_ctx / 32) + my_row / 32) * (4 * kDB)) * 256 + lane * 4;
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        floatx4 t;
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = acc[db][rg * 4 + c];
        __builtin_nontemporal_store(t, reinterpret_cast<floatx4*>(af + (db * 4 + rg) * 256));
      }
    if (pool) {
      // Mean-pooling of the work-group's raw queries (brought into the idle tile buffer by the last tile's load slots) and
      // of its anchors: float32 sums over block_size rows in ascending row order, divided by block_size, rounded to
      // bf16 - the same operations in the same order as pool_kernel, so the results are the same bit for bit.
      const int pbuf = n_tiles & 1;  // where the queries went
      float* mlds = reinterpret_cast<float*>(tiles.k[pbuf ^ 1]);
      if (half == 0) mlds[wave * 32 + c32] = m_run;
      __syncthreads();
      const int bs = p.block_size, n_pooled = BM / bs;  // pooled rows of this work-group (1 for block_size 128)
      const int n_pr = p.n_ctx / bs;
      const float d = (float)bs;
      if (tid < D) {
        // waves 0 and 1: one head-dim column per thread (the ordered sum is a serial chain per column, so the shorter
        // the chain per thread the sooner the work-group retires)
        for (int pp = 0; pp < n_pooled; ++pp) {
          float a0 = 0.f;
          for (int r0 = pp * bs; r0 < (pp + 1) * bs; r0 += 16) {  // 16 rows at a time (never across the K/V halves): reads first, then the ordered sums
            const char* rowp = (r0 < 64 ? tiles.k[pbuf] : tiles.v[pbuf]) + (r0 & 63) * kRowBytes + 2 * tid;
            uint16_t w[16];
#pragma unroll
            for (int t = 0; t < 16; ++t) w[t] = *reinterpret_cast<const uint16_t*>(rowp + t * kRowBytes);
#pragma unroll
            for (int t = 0; t < 16; ++t) a0 += T::from16(w[t]);
          }
          reinterpret_cast<uint16_t*>(p.qbar_out)[((bh * n_pr) + R0 / bs + pp) * D + tid] = (uint16_t)(T::pack(a0 / d, 0.f) & 0xffffu);
        }
      } else if (wave == 2) {
        // meanwhile, in wave 2: the pooled anchors, with all 64 lanes shared among them, and their thresholds
        const int lanes = 64 / n_pooled, pp = lane / lanes;
        float am = 0.f;
        for (int r0 = pp * bs; r0 < (pp + 1) * bs; r0 += 16) {
          float w[16];
#pragma unroll
          for (int t = 0; t < 16; t += 4) *reinterpret_cast<floatx4*>(&w[t]) = *reinterpret_cast<const floatx4*>(&mlds[r0 + t]);
#pragma unroll
          for (int t = 0; t < 16; ++t) am += w[t];
        }
        const uint32_t a16 = T::pack(am / d, 0.f) & 0xffffu;
        const int64_t row = bh * n_pr + R0 / bs + pp;
        if (lane % lanes == 0) reinterpret_cast<uint16_t*>(p.abar_out)[row] = (uint16_t)a16;
        if (p.thr_out != nullptr) {
          const uint32_t x = select_threshold<T>(T::from16((uint16_t)a16), p.scale2, p.theta_log2, lane, lanes);
          if (lane % lanes == 0) p.thr_out[row] = x;
        }
      }
    }
  } else if (kAnyRows && p.n_chunks > 1) {
    // one of several chunks: the unnormalised state goes to the workspace, in fragment order as in anchor mode, and
    // rows_combine_kernel merges the chunks
    const int64_t slot = ((((int64_t)b * p.n_kv_heads + kvh) * p.n_col_blocks + qunit) * p.n_chunks + chunk) * 4 + wave;
    if (half == 0) {
      p.M_out[slot * 32 + c32] = m_run;
      p.L_out[slot * 32 + c32] = l_tot;
    }
    float* af = p.acc_out + slot * (kDB * 4 * 256) + lane * 4;
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        floatx4 t;
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = acc[db][rg * 4 + c];
        *reinterpret_cast<floatx4*>(af + (db * 4 + rg) * 256) = t;
      }
  } else {
    // out = bf16(acc / l): the wave stages its [32][D] tile in LDS - 32 rows of the tile pitch, 16-byte chunks swizzled
    // with the row like a K tile - and writes whole rows.  The staging area is private to the wave (only a wave-local wait
    // lies between its writes and its reads) and lies in the tile buffer the loop consumed last, which every wave has
    // finished reading (the tile's closing barrier): waves 0, 1 in its K half, waves 2, 3 in its V half.  In sparse mode
    // the other buffer may already hold the next block's first tile.
    const bool more = MODE == kSparse && qb + 1 < nq;
    if (more) request_queries(my_row + BM);  // (the registers of this block's raw queries are long free)
    char* ob = (MODE == kSparse ? (wave < 2 ? tiles.k[cur ^ 1] : tiles.v[cur ^ 1]) + (wave & 1) * 32 * kRowBytes
                                : tiles.k[0] + wave * 32 * kRowBytes);
    constexpr int kChunkMask = D / 8 - 1;
    // (the staging offsets are the same for every block of the work-group; computed from an opaque copy of the lane
    // number they are formed here, a few instructions per block, instead of occupying registers throughout the tile loop)
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    const int c32_e = lane_e & 31, half_e = lane_e >> 5;
    const float inv = MODE == kMasked && l_tot == 0.f ? 0.f : 1.0f / l_tot;  // (a row that sees no key gives 0)
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        u32x2 w;
        w[0] = T::pack(acc[db][rg * 4 + 0] * inv, acc[db][rg * 4 + 1] * inv);
        w[1] = T::pack(acc[db][rg * 4 + 2] * inv, acc[db][rg * 4 + 3] * inv);
        *reinterpret_cast<u32x2*>(ob + c32_e * kRowBytes + (((4 * db + rg) ^ (c32_e & kChunkMask)) << 4) + 8 * half_e) = w;
      }
    // the accumulator registers are free: the next block's state can be on its way while this block's output leaves
    if (more && list_chains) request_state(my_row + BM);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's LDS writes are done (and stay above this line)
    uint16_t* op = p.out + b * p.o_sb + hq * p.o_sh;
    constexpr int kLanesPerRow = D / 8, kRowsPerStore = 64 / kLanesPerRow;  // a row is D/8 pieces of 16 bytes
#pragma unroll
    for (int it = 0; it < 32 / kRowsPerStore; ++it) {
      const int r = it * kRowsPerStore + lane_e / kLanesPerRow, c = lane_e % kLanesPerRow;
      const u32x4 w = *reinterpret_cast<const u32x4*>(ob + r * kRowBytes + ((c ^ (r & kChunkMask)) << 4));
      if (kAnyRows) {
        const int col = wr0 + r, row = (int)quotient((uint32_t)col, p.by_group);
        if (col < n_cols) *reinterpret_cast<u32x4*>(op + (col - row * group) * p.o_sh + (int64_t)row * p.o_sn + 8 * c) = w;
      } else {
        __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(op + (int64_t)(wr0 + r) * p.o_sn + 8 * c));
      }
    }
    chained = more && list_chains;
    have_queries = more;
    if (MODE == kAnchor && R0 == 0 && tid == 0 && p.zero_counts != nullptr) p.zero_counts[bh] = 0;  // (a single big block: nothing is selected)
  }
  }  // query blocks of the work-group
}

template <int MODE, typename T, int D, int TEAMS>
__global__ void __launch_bounds__(256 * TEAMS, TEAMS > 1 ? 1 : D == 128 ? 2 : 3) flash_kernel(const FlashArgs p) {
  __shared__ __attribute__((aligned(16))) FlashSmem<MODE, D, TEAMS> sm;
  flash_body<MODE, T, D, TEAMS>(p, blockIdx.x, sm);
}

// Anchor mode and rows mode in one launch, for a prompt that ends in part of a big block: the rows of that part depend on no other
// stage.  The rows' work-groups come first; anchor work-groups, longest first, fill the CUs beside and after them, so that the
// uneven end of one launch is the other's work and the rows need fewer key chunks to fill the chip - often none, and then no merge.
// The first anchor work-group's number is a multiple of 8: both bodies' maps from work-groups to XCDs hold.
// One launch against two, whole prompts: 32/8 heads of 128, 2200 tokens 68.5 -> 55.0 us, 3148 138 -> 109, 6001 375 -> 353, 40001 2955 -> 2878; 32/8
// heads of 64, 6001 230 -> 207; 14/2 heads of 64, 2600 44.3 -> 31.9, 7500 165 -> 142, 30000 630 -> 600.
template <typename T, int D, int TEAMS>
__global__ void __launch_bounds__(256 * TEAMS, TEAMS > 1 ? 1 : D == 128 ? 2 : 3)
flash_pair_kernel(const FlashArgs anchor, const FlashArgs rows, const uint32_t n_rows_wgs) {
  __shared__ __attribute__((aligned(16))) union {
    FlashSmem<kAnchor, D, TEAMS> anchor;
    FlashSmem<kRows, D, TEAMS> rows;
  } sm;
  const uint32_t n_first = (n_rows_wgs + 7u) & ~7u;
  if (blockIdx.x >= n_first) flash_body<kAnchor, T, D, TEAMS>(anchor, blockIdx.x - n_first, sm.anchor);
  else if (blockIdx.x < n_rows_wgs) flash_body<kRows, T, D, TEAMS>(rows, blockIdx.x, sm.rows);
}

#ifndef AA_SPARSE_QBLOCKS
#define AA_SPARSE_QBLOCKS 4  // most 128-row query blocks a stage-3 work-group handles one after the other
#endif

// Sets what the launcher decides for a launch of one mode, alone or with another; the number of work-groups.
template <int MODE>
static uint32_t place(FlashArgs& a, const bool alone) {
  set_heads(a);
  int64_t blocks = (int64_t)a.batch * a.n_q_heads * (a.n_ctx / 128);
  if (MODE == kSparse) {
    const int per_big_block = a.big_block / 128;
    a.n_big = a.n_ctx / a.big_block;
    blocks -= (int64_t)a.batch * a.n_q_heads * a.first_big_block * per_big_block;
    if (blocks == 0) return 0;
    // Chained blocks save a work-group's start and the list's round trip, but few work-groups leave CUs idle: as many as
    // still fill the chip twice (two work-groups per CU at head dimension 128, three at 64).  Four at any size against this
    // rule, operator: 14/2 heads of 64, 8192 tokens, every key selected 491 -> 288 us; 32/8 heads of 128, 4096 tokens
    // 353 -> 288 us, 16384 tokens 2661 -> 2568 us (filling the chip once: 2649); 32768 tokens, few keys: within 0.3 %.
    const int fills_twice = 2 * (a.head_dim == 128 ? 512 : 768);
    int nq = AA_SPARSE_QBLOCKS;
    while (nq > 1 && (per_big_block % nq != 0 || blocks / nq < fills_twice)) nq /= 2;
    a.q_blocks_per_wg = nq;
    a.q_units = per_big_block / nq;
    a.pairs = (int64_t)a.units * (a.n_big - a.first_big_block) % 8 == 0;
    if (a.pairs) {
      a.by_pair = fast_div(a.group * a.q_units);
      a.by_units = fast_div(a.units);
    } else {
      a.by_block = fast_div(a.q_units);
      a.deal = make_deal(a.units, a.group * (a.n_big - a.first_big_block) * a.q_units, a.group, false);
    }
    return (uint32_t)(blocks / nq) + (a.ratio != nullptr ? 1 : 0);
  } else if (MODE == kAnchor) {
    a.by_block = fast_div(a.big_block / 128);
  }
  // More units (KV heads of all batch elements) than XCDs: side by side as long as the K and V that an XCD then works on fit its L2
  // of 4 MB.  Left-padded batches: 3 x 2500 with 32/8 heads of 128 194 -> 184 us, 28/4 184 -> 162, 3 x 1000 with 32/8 heads of 64 39.9 -> 30.0, 4 x 2900
  // 162 -> 150; the operator on 2 x 4096 tokens with those heads 181 -> 172.  Larger contexts, where the order hardly matters: within 1 %.
  // So also fewer units than XCDs whose rows a unit's XCDs cannot share evenly (an odd number with 4 units): the hardware order ended with the heaviest
  // work-groups of the last unit.  1578 rows, 14/2 heads of 64 28.0 -> 23.3 us; padded 2 x 1920 48.5 -> 42.8; dense 4864 tokens 90.1 -> 69.3; with 28/4
  // heads of 128 1501 rows in one chunk 54.2 -> 41.3, dense 3712 fp16 142.5 -> 120.3.  A launch that anchor and rows work-groups share gains
  // nothing on average (44 sizes: from 10 % faster to 10 % slower).
  const int units = a.units;
  const int rows = MODE == kRows || MODE == kMasked ? a.n_col_blocks * a.n_chunks : a.n_ctx / 128;  // (of a unit: what is dealt out)
  const bool abreast = 8 % units != 0 ? (int64_t)((units + 7) / 8) * a.n_ctx * a.head_dim * 4 <= 4 << 20 : alone && rows % (8 / units) != 0;
  if (MODE == kRows || MODE == kMasked) {
    a.by_cols = fast_div(a.n_col_blocks);
    a.deal = make_deal(units, rows, 1, abreast);
    return (uint32_t)units * rows;
  }
  a.deal = make_deal(units, a.group * rows, a.group, abreast);
  return (uint32_t)blocks;
}

template <int MODE>
static int teams_of(const FlashArgs& a, const uint32_t work_groups) {
  // Two teams where a work-group is alone on its CU and its tiles pay for the merge (1.5 us).  Head dimension 64: 2048 tokens with 14/2
  // heads, one launch, 26.4 -> 22.9 us, dense 25.9 -> 22.3, 1024 tokens dense 15.0 -> 14.1, a prompt of 2348 44.3 -> 40.4, padded 2 x 1000 25.7 -> 23.3;
  // 512 tokens dense (8 tiles) 9.6 -> 10.2, and 512 work-groups (32 heads, 2048 tokens) 27.6 -> 29.5.
  // (anchor: a single big block only, whose rows are finished or leave their state; larger contexts give the same bits in any batch)
  const bool fits = MODE == kAnchor ? a.n_ctx == a.big_block && (a.qbar_out == nullptr || a.out != nullptr) : MODE != kSparse;
  return a.head_dim == 64 && fits && work_groups <= 256 && (MODE == kRows || MODE == kMasked ? a.chunk_tiles : a.n_ctx / kBN) >= 12 ? 2 : 1;
}

template <int MODE, typename T>
static void launch_for(const FlashArgs& a, const uint32_t work_groups, hipStream_t stream) {
  const dim3 grid(work_groups);
  if (a.head_dim == 128) hipLaunchKernelGGL((flash_kernel<MODE, T, 128, 1>), grid, dim3(256), 0, stream, a);
  else if (teams_of<MODE>(a, work_groups) == 1) hipLaunchKernelGGL((flash_kernel<MODE, T, 64, 1>), grid, dim3(256), 0, stream, a);
  else if constexpr (MODE != kSparse) hipLaunchKernelGGL((flash_kernel<MODE, T, 64, 2>), grid, dim3(512), 0, stream, a);
}

template <int MODE>
static hipError_t launch(FlashArgs a, hipStream_t stream) {
  const uint32_t work_groups = place<MODE>(a, true);
  if (work_groups == 0) return hipSuccess;
  if (a.dtype == 0) launch_for<MODE, Bf16>(a, work_groups, stream);
  else launch_for<MODE, F16>(a, work_groups, stream);
  return hipGetLastError();
}

template <typename T>
static void launch_pair_for(const FlashArgs& a, const FlashArgs& r, const uint32_t n_anchor, const uint32_t n_rows, hipStream_t stream) {
  const uint32_t both = ((n_rows + 7u) & ~7u) + n_anchor;
  const dim3 grid(both);
  if (a.head_dim == 128) hipLaunchKernelGGL((flash_pair_kernel<T, 128, 1>), grid, dim3(256), 0, stream, a, r, n_rows);
  else if (teams_of<kAnchor>(a, both) == 1 || teams_of<kRows>(r, both) == 1)
    hipLaunchKernelGGL((flash_pair_kernel<T, 64, 1>), grid, dim3(256), 0, stream, a, r, n_rows);
  else hipLaunchKernelGGL((flash_pair_kernel<T, 64, 2>), grid, dim3(512), 0, stream, a, r, n_rows);
}

hipError_t launch_anchor_and_rows(FlashArgs anchor, FlashArgs rows, hipStream_t stream) {
  const uint32_t n_anchor = place<kAnchor>(anchor, false), n_rows = place<kRows>(rows, false);
  if (anchor.dtype == 0) launch_pair_for<Bf16>(anchor, rows, n_anchor, n_rows, stream);
  else launch_pair_for<F16>(anchor, rows, n_anchor, n_rows, stream);
  return hipGetLastError();
}

hipError_t launch_flash(const FlashArgs& a, int mode, hipStream_t stream) {
  if (mode == kAnchor) return launch<kAnchor>(a, stream);
  if (mode == kSparse) return launch<kSparse>(a, stream);
  if (mode == kRows) return launch<kRows>(a, stream);
  if (mode == kMasked) return launch<kMasked>(a, stream);
  return launch<kDense>(a, stream);
}

}  // namespace aa
