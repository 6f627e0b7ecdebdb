// Internal launch interfaces between the C-ABI layer and the kernel translation units.
#pragma once
#include "aa_common.h"

namespace aa {

struct FlashArgs {
  const uint16_t* q; int64_t q_sb, q_sh, q_sn;
  const uint16_t* k; int64_t k_sb, k_sh, k_sn;
  const uint16_t* v; int64_t v_sb, v_sh, v_sn;
  uint16_t* out;     int64_t o_sb, o_sh, o_sn;   // all modes (anchor mode, optional: the first big block's rows, which select no keys, are finished there)
  float* M_out; float* L_out; float* acc_out;  // anchor mode
  // anchor mode, optional (both or neither; block_size <= 128): the work-group also mean-pools its 128 raw query rows
  // and anchors into qbar [B,Hq,N/block_size,head_dim] and abar [B,Hq,N/block_size], bit for bit what pool_kernel computes
  uint16_t* qbar_out; uint16_t* abar_out;
  // ... and, where it pools, the selection thresholds of its pooled rows (aa_threshold.h) into thr_out [B,Hq,N/block_size]
  uint32_t* thr_out; float scale2, theta_log2;
  // anchor mode, optional: [B,Hq], set to 0 where big block 0 is finished (the only one: nobody else writes its counts)
  int32_t* zero_counts;
  uint64_t* clear;  // anchor mode, optional: a word that is set to 0 (SelectArgs::selected)
  // anchor and sparse mode, optional: the ratio of selected keys, sum(counts[0 .. n_ratio_counts)) * ratio_inverse (anchor: 0)
  float* ratio; int64_t n_ratio_counts; float ratio_inverse;
  float* ratio_host;  // the same number in host memory, for a caller that waits for it and not for the launch to end
  const float* M; const float* L; const float* acc_frag;  // sparse mode (resume state)
  const int32_t* coords; const int32_t* counts; int64_t coords_per_head;  // sparse mode
  int batch, n_q_heads, n_kv_heads, n_ctx;
  int head_dim;  // 128 or 64
  int big_block, block_size;
  int first_big_block;  // sparse mode: 1 leaves out the rows of big block 0 (anchor mode has finished them), 0 takes all rows
  float sm_scale; int scale_mode;
  // set by the launchers
  int q_blocks_per_wg;
  Deal deal;        // which work-group has which rows
  int group;        // query heads of a KV head
  int units;        // KV heads of all batch elements
  int n_big;        // (sparse) big blocks
  int q_units;      // (sparse) work-groups of a big block and query head
  bool pairs;       // (sparse) (KV head, big block) pairs go round-robin
  FastDiv by_group, by_kv_heads;
  FastDiv by_cols;    // (rows, masked) column blocks; (merge of a decode step) columns
  FastDiv by_chunks;  // (decode) chunks; (merge of rows) tiles of a chunk
  FastDiv by_block;   // (anchor, sparse) work-groups of a big block and query head
  FastDiv by_pair, by_units;  // (sparse, pairs) work-groups of a (KV head, big block) pair; KV heads of all batch elements
  // rows mode: n_rows query rows over n_ctx keys, row i sees keys 0 .. causal_offset + i.  The (row, head) columns of a
  // KV head come in blocks of 128, the keys in chunks of chunk_tiles 64-key tiles; with more than one chunk the work-groups
  // write M_out, L_out, acc_out [batch, n_kv_heads, n_col_blocks, n_chunks, 128 columns] for rows_combine_kernel
  int n_rows, causal_offset, n_col_blocks, n_chunks, chunk_tiles;
  // masked mode (rows mode whose causal_offset lets every row see every key, and a boolean mask): the mask as bits
  // [batch, n_rows, mask_words_per_row] (bit j of word t: key 64 t + j), and what each tile of each column block holds,
  // tile_flags [batch, n_col_blocks, mask_words_per_row]: 0 nothing visible, 1 some, 2 every key to every row
  const uint64_t* mask_words; const uint8_t* tile_flags; int mask_words_per_row;
  int decode_waves;  // decode kernel: waves of a work-group, 4 or 1
  // decode kernel with a mask (one query row): the byte mask itself
  const uint8_t* mask_bytes; int64_t mask_sb;
  int dtype;            // AA_DTYPE_BF16 / AA_DTYPE_F16: what the 16-bit elements of q, k, v, out, qbar, abar are
};

// what all kernels find their place by
inline void set_heads(FlashArgs& a) {
  a.group = a.n_q_heads / a.n_kv_heads;
  a.units = a.batch * a.n_kv_heads;
  a.by_group = fast_div(a.group);
  a.by_kv_heads = fast_div(a.n_kv_heads);
}

// mode: 0 anchor (stage 1), 1 sparse (stage 3), 2 dense causal, 3 rows, 4 masked
hipError_t launch_flash(const FlashArgs& a, int mode, hipStream_t stream);
// anchor mode and rows mode (same types and head dimension) in one launch
hipError_t launch_anchor_and_rows(FlashArgs anchor, FlashArgs rows, hipStream_t stream);

// rows mode with several chunks: merges the chunks of `a` (the arguments of the launch that wrote them) into a.out
hipError_t launch_rows_combine(FlashArgs a, hipStream_t stream);
// rows mode: sets n_col_blocks, n_chunks and chunk_tiles from the sizes and the type
void plan_rows(FlashArgs& a);
// ... for a launch that anchor work-groups of `anchor` share (launch_anchor_and_rows)
void plan_rows_beside(FlashArgs& a, const FlashArgs& anchor);
constexpr int kMaskedTiles = 1024;  // most tiles in a chunk of masked mode (the list of a chunk's visible tiles lives in LDS)
// masked mode: fills mask_words and tile_flags of `a` from a byte mask [batch, n_rows, n_ctx] with strides (mask_sb, mask_sn, 1)
hipError_t launch_mask_pack(const FlashArgs& a, const uint8_t* mask, int64_t mask_sb, int64_t mask_sn, hipStream_t stream);

// A few query rows over many keys (decode steps): the arguments of rows mode, one column block, chunk_tiles counted in 32-key
// tiles, and the chunks' state as M_out, L_out [batch, n_kv_heads, n_chunks, columns] and acc_out [..., columns, head_dim].
constexpr int kDecMaxChunks = 256;
bool decode_takes(int n_rows, int group, bool masked);
void plan_decode(FlashArgs& a);
hipError_t launch_decode(FlashArgs& a, hipStream_t stream);

// x, out [rows, hidden], weight [hidden], contiguous; hidden a multiple of 8 and at most 16384
hipError_t launch_rms_norm(const uint16_t* x, const uint16_t* weight, uint16_t* out, int64_t rows, int hidden, float eps, int dtype, hipStream_t stream);
// n elements, a multiple of 8
hipError_t launch_silu_mul(const uint16_t* gate, const uint16_t* up, uint16_t* out, int64_t n, int dtype, hipStream_t stream);

// queries [batch, n_q_heads, n_tokens, head_dim] and keys with n_kv_heads, rotated into q_out and k_out; cos, sin [batch or 1 (cs_sb 0), n_tokens, head_dim]
struct RopeArgs {
  const uint16_t* q; int64_t q_sb, q_sh, q_sn;
  const uint16_t* k; int64_t k_sb, k_sh, k_sn;
  uint16_t* q_out; int64_t qo_sb, qo_sh, qo_sn;
  uint16_t* k_out; int64_t ko_sb, ko_sh, ko_sn;
  const uint16_t* cos; const uint16_t* sin; int64_t cs_sb;
  int batch, n_q_heads, n_kv_heads, n_tokens, head_dim;  // a multiple of 16; fewer than 2^32 threads
};
hipError_t launch_rope(const RopeArgs& a, int dtype, hipStream_t stream);

struct PoolArgs {
  const uint16_t* q; int64_t q_sb, q_sh, q_sn;
  const float* M;
  uint16_t* qbar; uint16_t* abar;
  int batch, n_q_heads, n_ctx, block_size;
  int head_dim;  // 128 or 64
  int dtype;
};
hipError_t launch_pool(const PoolArgs& a, hipStream_t stream);

struct SelectArgs {
  const uint16_t* qbar; const uint16_t* abar;
  const uint16_t* k; int64_t k_sb, k_sh, k_sn;
  float* thr;  // per pooled row: smallest raw dot product that passes the selection test
  uint32_t* mask; int32_t* coords; int32_t* counts; int64_t coords_per_head;
  int batch, n_q_heads, n_kv_heads, n_ctx;
  int big_block, block_size;
  float scale2, theta_log2;
  // optional: the share of selected keys, formed by the work-groups of the scores as in FlashArgs; `selected` is 0 before
  uint64_t* selected; float* ratio; float* ratio_host; float ratio_inverse;
  // candidate keys of big block bb: key_lo <= j < bb*S - key_slack (as run: block_size and block_size; intended: S and 0)
  int key_lo, key_slack;
  int head_dim;  // 128 or 64
  int dtype;
  // set by the launcher of the scores: which work-group has which keys
  Deal deal; FastDiv by_kv_heads;
};
hipError_t launch_select_thresholds(const SelectArgs& a, hipStream_t stream);
hipError_t launch_select_scores(SelectArgs a, hipStream_t stream);
bool select_scores_sums(int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim, int big_block);  // whether that is to form the ratio
hipError_t launch_select_compact(const SelectArgs& a, hipStream_t stream);
hipError_t launch_ratio(const int32_t* counts, int64_t n, float inverse, float* ratio, hipStream_t stream);

}  // namespace aa
