// C ABI of the AnchorAttention gfx950 kernels: argument validation, scratch carving, launches.
// Declarations and their reference counterparts: include/anchor_attn_hip.h.
#include <algorithm>
#include <chrono>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "../../include/anchor_attn_hip.h"
#include "aa_common.h"
#include "aa_kernels.h"

// Device memory for aa_stage2_select_static(): the stage-2 bitmask and thresholds of callers that cannot
// allocate.  Every GPU the library's code object is loaded on holds its own copy until the process ends.  In host
// code this name only stands for the symbol; the memory's address on a device comes from hipGetSymbolAddress().
static __device__ __align__(256) unsigned char scratch[AA_STATIC_SCRATCH_BYTES];

namespace aa {

static thread_local char g_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

namespace {

struct Dims {
  int batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step;
};

// Checks every entry point shares: head counts, head_dim, and the sizes one launch can address.
int check_common_dims(const Dims& d, const char* who) {
  if (d.batch <= 0 || d.n_q_heads <= 0 || d.n_kv_heads <= 0 || d.n_ctx <= 0) {
    set_error("%s: batch, head counts and n_ctx must be positive (got %d, %d, %d, %d)", who, d.batch, d.n_q_heads, d.n_kv_heads, d.n_ctx);
    return AA_EBADARG;
  }
  if (d.n_q_heads % d.n_kv_heads != 0) {
    set_error("%s: n_kv_heads (%d) must divide n_q_heads (%d)", who, d.n_kv_heads, d.n_q_heads);
    return AA_EBADARG;
  }
  if (d.head_dim != 128 && d.head_dim != 64) {
    set_error("%s: head_dim %d is not supported (128 or 64)", who, d.head_dim);
    return AA_EUNSUPPORTED;
  }
  if (d.n_ctx % 128 != 0) {
    set_error("%s: n_ctx %d must be a multiple of 128", who, d.n_ctx);
    return AA_EUNSUPPORTED;
  }
  if (d.n_ctx > (1 << 20)) {
    set_error("%s: n_ctx %d is larger than 1048576", who, d.n_ctx);
    return AA_EUNSUPPORTED;
  }
  if ((int64_t)d.batch * d.n_q_heads * (d.n_ctx / 128) > 0x7fffffffLL) {
    set_error("%s: problem too large for one launch", who);
    return AA_EUNSUPPORTED;
  }
  return AA_OK;
}

// The common checks plus the big-block geometry of the three AnchorAttention stages.
int check_dims(const Dims& d, const char* who) {
  if (int rc = check_common_dims(d, who)) return rc;
  if (d.block_size != 16 && d.block_size != 32 && d.block_size != 64 && d.block_size != 128 && d.block_size != 256) {
    set_error("%s: block_size %d is not supported (16, 32, 64, 128 or 256)", who, d.block_size);
    return AA_EUNSUPPORTED;
  }
  if (d.step != 16 && d.step != 32) {
    set_error("%s: step %d is not supported (16 or 32)", who, d.step);
    return AA_EUNSUPPORTED;
  }
  if (d.n_ctx % (d.block_size * d.step) != 0) {
    set_error("%s: n_ctx %d is not a multiple of block_size*step = %d", who, d.n_ctx, d.block_size * d.step);
    return AA_EUNSUPPORTED;
  }
  return AA_OK;
}

// What stage 2 asks beyond that: the score kernel numbers (query head of the KV group, big block) pairs with 16 bits and
// addresses the pooled queries with 32-bit byte offsets.
int check_select(const Dims& d, int geometry, const char* who) {
  if (geometry != AA_GEOMETRY_AS_RUN && geometry != AA_GEOMETRY_INTENDED) {
    set_error("%s: geometry %d is neither AA_GEOMETRY_AS_RUN nor AA_GEOMETRY_INTENDED", who, geometry);
    return AA_EBADARG;
  }
  if ((int64_t)(d.n_q_heads / d.n_kv_heads) * (d.n_ctx / (d.block_size * d.step)) >= 65536 ||
      (int64_t)d.batch * d.n_q_heads * (d.n_ctx / d.block_size) * 2 * d.head_dim > 0xffffffffLL) {
    set_error("%s: too many (head, big block) pairs or pooled rows for one launch (heads per KV head %d, big blocks %d, pooled rows %lld)",
              who, d.n_q_heads / d.n_kv_heads, d.n_ctx / (d.block_size * d.step), (long long)d.batch * d.n_q_heads * (d.n_ctx / d.block_size));
    return AA_EUNSUPPORTED;
  }
  return AA_OK;
}

int check_tensor(const void* ptr, int64_t sb, int64_t sh, int64_t sn, int n_ctx, int head_dim, const char* who, const char* name) {
  if (ptr == nullptr) {
    set_error("%s: %s is NULL", who, name);
    return AA_EBADARG;
  }
  if ((reinterpret_cast<uintptr_t>(ptr) & 15u) != 0 || (sb % 8) != 0 || (sh % 8) != 0 || (sn % 8) != 0) {
    set_error("%s: %s must be 16-byte aligned with strides that are multiples of 8 elements (ptr=%p strides=%lld,%lld,%lld)", who, name, ptr, (long long)sb, (long long)sh, (long long)sn);
    return AA_EMISALIGNED;
  }
  if (sn < head_dim) {
    set_error("%s: %s row stride %lld is smaller than head_dim", who, name, (long long)sn);
    return AA_EBADARG;
  }
  if (sn > (int64_t)1 << 14) {  // the kernels address rows of one head with 32-bit byte offsets
    set_error("%s: %s row stride %lld is larger than 16384 elements", who, name, (long long)sn);
    return AA_EUNSUPPORTED;
  }
  if ((int64_t)n_ctx * sn * 2 > (int64_t)0xffffffffLL) {
    set_error("%s: %s spans %lld bytes per head (n_ctx %d x row stride %lld elements); the kernels address one head with 32-bit byte offsets",
              who, name, (long long)n_ctx * sn * 2, n_ctx, (long long)sn);
    return AA_EUNSUPPORTED;
  }
  return AA_OK;
}

int check_ptr(const void* ptr, const char* who, const char* name) {
  if (ptr == nullptr) {
    set_error("%s: %s is NULL", who, name);
    return AA_EBADARG;
  }
  if ((reinterpret_cast<uintptr_t>(ptr) & 15u) != 0) {
    set_error("%s: %s must be 16-byte aligned", who, name);
    return AA_EMISALIGNED;
  }
  return AA_OK;
}

int check_dtype(int dtype, const char* who) {
  if (dtype != AA_DTYPE_BF16 && dtype != AA_DTYPE_F16) {
    set_error("%s: dtype %d is neither AA_DTYPE_BF16 nor AA_DTYPE_F16", who, dtype);
    return AA_EBADARG;
  }
  return AA_OK;
}

int check_launch(hipError_t e, const char* who) {
  if (e != hipSuccess) {
    set_error("%s: launch failed: %s", who, hipGetErrorString(e));
    return AA_ELAUNCH;
  }
  return AA_OK;
}

hipError_t run_flash(const FlashArgs& a, int mode, hipStream_t stream) {
  return launch_flash(a, mode, stream);
}

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// Address of `scratch` on the current device, looked up once per device (with that device current) and kept.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

int static_scratch(void** out, const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("%s: cannot tell the current device (%s, device %d)", who, hipGetErrorString(e), dev);
    return AA_ELAUNCH;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      set_error("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", who, dev, hipGetErrorString(e));
      return AA_ELAUNCH;
    }
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return AA_OK;
}

struct Workspace {
  size_t M, L, acc, qbar, abar, mask, coords, counts, total;
};

Workspace carve(int batch, int hq, int n_ctx, int head_dim, int block_size, int step) {
  Workspace w;
  const size_t bh = (size_t)batch * hq;
  size_t off = 0;
  w.M = off;      off += align256(bh * n_ctx * 4);
  w.L = off;      off += align256(bh * n_ctx * 4);
  w.acc = off;    off += align256(bh * n_ctx * head_dim * 4);
  w.qbar = off;   off += align256(bh * (n_ctx / block_size) * head_dim * 2);
  w.abar = off;   off += align256(bh * (n_ctx / block_size) * 2);
  w.mask = off;   off += align256((size_t)aa_mask_words(batch, hq, n_ctx, block_size, step) * 4);
  w.coords = off; off += align256(bh * (size_t)aa_coords_entries_per_head(n_ctx, block_size, step) * 4);
  w.counts = off; off += align256(bh * (n_ctx / (block_size * step)) * 4);
  w.total = off;
  return w;
}

}  // namespace
}  // namespace aa

using namespace aa;

extern "C" {

int aa_version(void) { return 3; }

const char* aa_last_error(void) { return g_error; }

int64_t aa_coords_entries_per_head(int n_ctx, int block_size, int step) {
  const int64_t S = (int64_t)block_size * step;
  return coords_tri(n_ctx / S, S, block_size);
}

int64_t aa_coords_offset(int big_block, int block_size, int step) {
  return coords_tri(big_block, (int64_t)block_size * step, block_size);
}

static int64_t mask_bit_words(int batch, int n_q_heads, int n_ctx, int block_size, int step) {
  return (int64_t)batch * n_q_heads * (n_ctx / (block_size * step)) * (n_ctx / 128) * 4;
}

int64_t aa_mask_words(int batch, int n_q_heads, int n_ctx, int block_size, int step) {
  // key bitmask followed by one float32 threshold per pooled row
  return mask_bit_words(batch, n_q_heads, n_ctx, block_size, step) + (int64_t)batch * n_q_heads * (n_ctx / block_size);
}

size_t aa_workspace_bytes(int batch, int n_q_heads, int n_ctx, int head_dim, int block_size, int step) {
  if (batch <= 0 || n_q_heads <= 0 || n_ctx <= 0 || (head_dim != 128 && head_dim != 64) || block_size <= 0 || step <= 0) return 0;
  return carve(batch, n_q_heads, n_ctx, head_dim, block_size, step).total;
}

// The share of selected keys, their number times `inverse`, where it is wanted; `selected`: a word that is 0, where stage 2 is to form it.
struct Ratio {
  float* ratio; float* host; float inverse; uint64_t* selected;
};

// What stage 1 does for the stages after it in the whole operator.
struct Stage1Extras {
  void* qbar; void* abar;  // pooled queries and anchors (block_size <= 128)
  float* thr; float scale2, theta_log2;  // and the thresholds of the pooled rows
  // the output of big block 0, whose rows select no keys, in the place of their state and pooled rows
  void* out; int64_t o_sb, o_sh, o_sn;
  uint64_t* clear;  // Ratio::selected
  int32_t* zero_counts; float* zero_ratio; float* zero_ratio_host;  // a single big block: what the later stages would say
  const FlashArgs* rows;  // a rows-mode problem that shares the launch
};

static int stage1_impl(const char* who, const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                       const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                       const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                       float* M, float* L, float* acc_frag, const Stage1Extras& x, int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                       int block_size, int step, float sm_scale, int scale_mode, int dtype, void* stream) {
  int rc;
  if ((rc = check_dims({batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step}, who))) return rc;
  if ((rc = check_dtype(dtype, who))) return rc;
  if ((rc = check_tensor(q, q_sb, q_sh, q_sn, n_ctx, head_dim, who, "q"))) return rc;
  if ((rc = check_tensor(k, k_sb, k_sh, k_sn, n_ctx, head_dim, who, "k"))) return rc;
  if ((rc = check_tensor(v, v_sb, v_sh, v_sn, n_ctx, head_dim, who, "v"))) return rc;
  if ((rc = check_ptr(M, who, "M")) || (rc = check_ptr(L, who, "L")) || (rc = check_ptr(acc_frag, who, "acc_frag"))) return rc;
  if (scale_mode != AA_SCALE_BF16_CHAIN && scale_mode != AA_SCALE_FP32) {
    set_error("%s: unknown scale_mode %d", who, scale_mode);
    return AA_EBADARG;
  }
  FlashArgs a = {};
  a.q = (const uint16_t*)q; a.q_sb = q_sb; a.q_sh = q_sh; a.q_sn = q_sn;
  a.k = (const uint16_t*)k; a.k_sb = k_sb; a.k_sh = k_sh; a.k_sn = k_sn;
  a.v = (const uint16_t*)v; a.v_sb = v_sb; a.v_sh = v_sh; a.v_sn = v_sn;
  a.M_out = M; a.L_out = L; a.acc_out = acc_frag;
  a.out = (uint16_t*)x.out; a.o_sb = x.o_sb; a.o_sh = x.o_sh; a.o_sn = x.o_sn;
  a.qbar_out = (uint16_t*)x.qbar; a.abar_out = (uint16_t*)x.abar;
  a.thr_out = reinterpret_cast<uint32_t*>(x.thr); a.scale2 = x.scale2; a.theta_log2 = x.theta_log2;
  a.clear = x.clear; a.zero_counts = x.zero_counts; a.ratio = x.zero_ratio; a.ratio_host = x.zero_ratio_host;
  a.batch = batch; a.n_q_heads = n_q_heads; a.n_kv_heads = n_kv_heads; a.n_ctx = n_ctx; a.head_dim = head_dim;
  a.big_block = block_size * step; a.block_size = block_size;
  a.sm_scale = sm_scale; a.scale_mode = scale_mode; a.dtype = dtype;
  if (x.rows != nullptr) return check_launch(launch_anchor_and_rows(a, *x.rows, (hipStream_t)stream), who);
  return check_launch(run_flash(a, 0, (hipStream_t)stream), who);
}

int aa_stage1_anchor_fwd(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                         const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                         const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                         float* M, float* L, float* acc_frag,
                         int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                         int block_size, int step, float sm_scale, int scale_mode, int dtype, void* stream) {
  return stage1_impl("aa_stage1_anchor_fwd", q, q_sb, q_sh, q_sn, k, k_sb, k_sh, k_sn, v, v_sb, v_sh, v_sn, M, L, acc_frag, Stage1Extras{},
                     batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step, sm_scale, scale_mode, dtype, stream);
}

int aa_pool_q_anchor(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn, const float* M,
                     void* qbar, void* abar,
                     int batch, int n_q_heads, int n_ctx, int head_dim, int block_size, int dtype, void* stream) {
  const char* who = "aa_pool_q_anchor";
  int rc;
  if ((rc = check_dtype(dtype, who))) return rc;
  if ((rc = check_dims({batch, n_q_heads, n_q_heads, n_ctx, head_dim, block_size, 16}, who))) return rc;
  if ((rc = check_tensor(q, q_sb, q_sh, q_sn, n_ctx, head_dim, who, "q"))) return rc;
  if ((rc = check_ptr(M, who, "M")) || (rc = check_ptr(qbar, who, "qbar")) || (rc = check_ptr(abar, who, "abar"))) return rc;
  PoolArgs a = {};
  a.q = (const uint16_t*)q; a.q_sb = q_sb; a.q_sh = q_sh; a.q_sn = q_sn;
  a.M = M; a.qbar = (uint16_t*)qbar; a.abar = (uint16_t*)abar;
  a.batch = batch; a.n_q_heads = n_q_heads; a.n_ctx = n_ctx; a.block_size = block_size; a.head_dim = head_dim; a.dtype = dtype;
  return check_launch(launch_pool(a, (hipStream_t)stream), who);
}

static float select_scale2(double sm_scale) { return (float)(sm_scale * 1.44269504); }  // double product, then float32, as the definition does

// Stage 2; have_thresholds: stage 1 has formed them.
static int stage2_impl(const char* who, bool have_thresholds, const Ratio& r, const void* qbar, const void* abar,
                     const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                     uint32_t* mask_ws, int32_t* coords, int32_t* counts,
                     int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                     int block_size, int step, double sm_scale, float theta_log2, int geometry, int dtype, void* stream) {
  int rc;
  if ((rc = check_dtype(dtype, who))) return rc;
  const Dims dims = {batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step};
  if ((rc = check_dims(dims, who)) || (rc = check_select(dims, geometry, who))) return rc;
  if ((rc = check_tensor(k, k_sb, k_sh, k_sn, n_ctx, head_dim, who, "k"))) return rc;
  if ((rc = check_ptr(qbar, who, "qbar")) || (rc = check_ptr(abar, who, "abar")) || (rc = check_ptr(mask_ws, who, "mask_ws")) ||
      (rc = check_ptr(coords, who, "coords")) || (rc = check_ptr(counts, who, "counts")))
    return rc;
  SelectArgs a = {};
  a.qbar = (const uint16_t*)qbar; a.abar = (const uint16_t*)abar;
  a.k = (const uint16_t*)k; a.k_sb = k_sb; a.k_sh = k_sh; a.k_sn = k_sn;
  a.mask = mask_ws; a.coords = coords; a.counts = counts;
  a.thr = reinterpret_cast<float*>(mask_ws + mask_bit_words(batch, n_q_heads, n_ctx, block_size, step));
  a.coords_per_head = aa_coords_entries_per_head(n_ctx, block_size, step);
  a.batch = batch; a.n_q_heads = n_q_heads; a.n_kv_heads = n_kv_heads; a.n_ctx = n_ctx; a.head_dim = head_dim;
  a.big_block = block_size * step; a.block_size = block_size;
  a.scale2 = select_scale2(sm_scale);
  a.theta_log2 = theta_log2;
  a.dtype = dtype;
  if (r.selected != nullptr) { a.selected = r.selected; a.ratio = r.ratio; a.ratio_host = r.host; a.ratio_inverse = r.inverse; }
  a.key_lo = geometry == AA_GEOMETRY_AS_RUN ? block_size : block_size * step;
  a.key_slack = geometry == AA_GEOMETRY_AS_RUN ? block_size : 0;
  if (n_ctx > block_size * step) {  // (a single big block has no candidates: its counts are 0)
    if (!have_thresholds && (rc = check_launch(launch_select_thresholds(a, (hipStream_t)stream), who))) return rc;
    if ((rc = check_launch(launch_select_scores(a, (hipStream_t)stream), who))) return rc;
  }
  return check_launch(launch_select_compact(a, (hipStream_t)stream), who);
}

int aa_stage2_select(const void* qbar, const void* abar,
                     const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                     uint32_t* mask_ws, int32_t* coords, int32_t* counts,
                     int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                     int block_size, int step, double sm_scale, float theta_log2, int geometry, int dtype, void* stream) {
  return stage2_impl("aa_stage2_select", false, Ratio{}, qbar, abar, k, k_sb, k_sh, k_sn, mask_ws, coords, counts, batch, n_q_heads, n_kv_heads, n_ctx,
                     head_dim, block_size, step, sm_scale, theta_log2, geometry, dtype, stream);
}

int aa_stage2_select_static(const void* qbar, const void* abar,
                            const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                            int32_t* coords, int32_t* counts,
                            int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                            int block_size, int step, double sm_scale, float theta_log2, int geometry, int dtype, void* stream) {
  const char* who = "aa_stage2_select_static";
  int rc;
  if ((rc = check_dims({batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step}, who))) return rc;
  const int64_t need = aa_mask_words(batch, n_q_heads, n_ctx, block_size, step) * 4;
  if (need > (int64_t)AA_STATIC_SCRATCH_BYTES) {
    set_error("%s: this problem needs %lld bytes of stage-2 scratch, the static scratch holds %lld (batch*n_q_heads*n_ctx^2 too "
              "large: use aa_stage2_select with a caller-provided buffer)", who, (long long)need, (long long)AA_STATIC_SCRATCH_BYTES);
    return AA_EUNSUPPORTED;
  }
  void* ws = nullptr;
  if ((rc = static_scratch(&ws, who))) return rc;
  // from here on exactly aa_stage2_select: same checks, same kernels, the scratch pointer as an ordinary argument
  return aa_stage2_select(qbar, abar, k, k_sb, k_sh, k_sn, static_cast<uint32_t*>(ws), coords, counts, batch, n_q_heads,
                          n_kv_heads, n_ctx, head_dim, block_size, step, sm_scale, theta_log2, geometry, dtype, stream);
}

// Stage 3 for the rows from big block `first_big_block` (0 or 1) on; also the ratio where stage 2 has not formed it.
static int stage3_impl(const char* who, int first_big_block, const Ratio& r,
                       const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                         const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                         const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                         const int32_t* coords, const int32_t* counts,
                         const float* M, const float* L, const float* acc_frag,
                         void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn,
                         int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                         int block_size, int step, float sm_scale, int dtype, void* stream) {
  int rc;
  if ((rc = check_dtype(dtype, who))) return rc;
  if ((rc = check_dims({batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step}, who))) return rc;
  if ((rc = check_tensor(q, q_sb, q_sh, q_sn, n_ctx, head_dim, who, "q"))) return rc;
  if ((rc = check_tensor(k, k_sb, k_sh, k_sn, n_ctx, head_dim, who, "k"))) return rc;
  if ((rc = check_tensor(v, v_sb, v_sh, v_sn, n_ctx, head_dim, who, "v"))) return rc;
  if ((rc = check_tensor(out, o_sb, o_sh, o_sn, n_ctx, head_dim, who, "out"))) return rc;
  if ((rc = check_ptr(coords, who, "coords")) || (rc = check_ptr(counts, who, "counts")) || (rc = check_ptr(M, who, "M")) ||
      (rc = check_ptr(L, who, "L")) || (rc = check_ptr(acc_frag, who, "acc_frag")))
    return rc;
  FlashArgs a = {};
  a.q = (const uint16_t*)q; a.q_sb = q_sb; a.q_sh = q_sh; a.q_sn = q_sn;
  a.k = (const uint16_t*)k; a.k_sb = k_sb; a.k_sh = k_sh; a.k_sn = k_sn;
  a.v = (const uint16_t*)v; a.v_sb = v_sb; a.v_sh = v_sh; a.v_sn = v_sn;
  a.out = (uint16_t*)out; a.o_sb = o_sb; a.o_sh = o_sh; a.o_sn = o_sn;
  a.M = M; a.L = L; a.acc_frag = acc_frag;
  a.coords = coords; a.counts = counts;
  a.coords_per_head = aa_coords_entries_per_head(n_ctx, block_size, step);
  a.batch = batch; a.n_q_heads = n_q_heads; a.n_kv_heads = n_kv_heads; a.n_ctx = n_ctx; a.head_dim = head_dim;
  a.big_block = block_size * step; a.block_size = block_size; a.first_big_block = first_big_block;
  a.sm_scale = sm_scale; a.scale_mode = AA_SCALE_FP32; a.dtype = dtype;
  if (r.selected == nullptr) { a.ratio = r.ratio; a.ratio_host = r.host; a.ratio_inverse = r.inverse; }
  a.n_ratio_counts = (int64_t)batch * n_q_heads * (n_ctx / a.big_block);
  return check_launch(run_flash(a, 1, (hipStream_t)stream), who);
}

int aa_stage3_sparse_fwd(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                         const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                         const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                         const int32_t* coords, const int32_t* counts,
                         const float* M, const float* L, const float* acc_frag,
                         void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn,
                         int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                         int block_size, int step, float sm_scale, int dtype, void* stream) {
  return stage3_impl("aa_stage3_sparse_fwd", 0, Ratio{}, q, q_sb, q_sh, q_sn, k, k_sb, k_sh, k_sn, v, v_sb, v_sh, v_sn, coords, counts, M, L, acc_frag,
                     out, o_sb, o_sh, o_sn, batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step, sm_scale, dtype, stream);
}

// The whole operator; with `ratio` the counts are kept in the workspace and their sum over `denominator` is formed.  `rows`: a rows-mode
// problem, checked and planned, that shares stage 1's launch.
static int anchor_attn_impl(const char* who, const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                       const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                       const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                       void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn,
                       void* workspace, size_t workspace_bytes, int32_t* counts_out, float* ratio, float* ratio_host, double denominator,
                       int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                       int block_size, int step, double sm_scale, float theta_log2, int scale_mode, int geometry,
                       int dtype, void* stream, const FlashArgs* rows = nullptr) {
  int rc;
  // (all that a later stage could refuse is looked at first: stage 1 already writes the first big block's output)
  const Dims dims = {batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step};
  if ((rc = check_dims(dims, who)) || (rc = check_select(dims, geometry, who))) return rc;
  if ((rc = check_ptr(workspace, who, "workspace"))) return rc;
  const Workspace w = carve(batch, n_q_heads, n_ctx, head_dim, block_size, step);
  if (workspace_bytes < w.total) {
    set_error("%s: workspace has %zu bytes, %zu needed", who, workspace_bytes, w.total);
    return AA_EBADARG;
  }
  char* ws = static_cast<char*>(workspace);
  float* M = (float*)(ws + w.M);
  float* L = (float*)(ws + w.L);
  float* acc = (float*)(ws + w.acc);
  void* qbar = ws + w.qbar;
  void* abar = ws + w.abar;
  uint32_t* mask = (uint32_t*)(ws + w.mask);
  int32_t* coords = (int32_t*)(ws + w.coords);
  // (stage 2 writes the counts where the caller wants them; a pointer that is not aligned for that gets a copy)
  const bool counts_direct = counts_out != nullptr && (reinterpret_cast<uintptr_t>(counts_out) & 15u) == 0;
  int32_t* counts = counts_direct ? counts_out : (int32_t*)(ws + w.counts);
  if ((rc = check_tensor(out, o_sb, o_sh, o_sn, n_ctx, head_dim, who, "out"))) return rc;
  // A stage-1 work-group holds 128 query rows: whole pooled rows when block_size <= 128, and then it pools them itself
  // (same arithmetic as aa_pool_q_anchor, bit for bit) and finds their thresholds instead of a pass over the queries and a launch.
  const bool fused_pool = block_size <= 128;
  // Big block 0 selects nothing and is finished by stage 1; stages 2 and 3 are for the others.
  const bool selects = n_ctx > block_size * step;
  Stage1Extras x = {};
  if (fused_pool) {
    x.qbar = qbar; x.abar = abar;
    x.thr = reinterpret_cast<float*>(mask + mask_bit_words(batch, n_q_heads, n_ctx, block_size, step));
    x.scale2 = select_scale2(sm_scale); x.theta_log2 = theta_log2;
  }
  x.out = out; x.o_sb = o_sb; x.o_sh = o_sh; x.o_sn = o_sn;
  x.rows = rows;
  // (the word for the sum lies where the lists will)
  const bool sums = selects && ratio != nullptr && select_scores_sums(batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size * step);
  const Ratio r = {ratio, ratio_host, 1.f / (float)denominator, sums ? reinterpret_cast<uint64_t*>(coords) : nullptr};
  x.clear = r.selected;
  if (!selects) { x.zero_counts = counts; x.zero_ratio = ratio; x.zero_ratio_host = ratio_host; }
  if ((rc = stage1_impl(who, q, q_sb, q_sh, q_sn, k, k_sb, k_sh, k_sn, v, v_sb, v_sh, v_sn, M, L, acc, x, batch, n_q_heads, n_kv_heads,
                        n_ctx, head_dim, block_size, step, (float)sm_scale, scale_mode, dtype, stream)))
    return rc;
  if (rows != nullptr && rows->n_chunks > 1 && (rc = check_launch(launch_rows_combine(*rows, (hipStream_t)stream), who))) return rc;
  if (selects) {
    if (!fused_pool &&
        (rc = aa_pool_q_anchor(q, q_sb, q_sh, q_sn, M, qbar, abar, batch, n_q_heads, n_ctx, head_dim, block_size, dtype, stream)))
      return rc;
    if ((rc = stage2_impl(who, fused_pool, r, qbar, abar, k, k_sb, k_sh, k_sn, mask, coords, counts, batch, n_q_heads, n_kv_heads, n_ctx,
                          head_dim, block_size, step, sm_scale, theta_log2, geometry, dtype, stream)))
      return rc;
    if ((rc = stage3_impl(who, 1, r, q, q_sb, q_sh, q_sn, k, k_sb, k_sh, k_sn, v, v_sb, v_sh, v_sn, coords, counts, M, L, acc,
                          out, o_sb, o_sh, o_sn, batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step, (float)sm_scale, dtype,
                          stream)))
      return rc;
  }
  if (counts_out != nullptr && !counts_direct) {
    const size_t bytes = (size_t)batch * n_q_heads * (n_ctx / (block_size * step)) * 4;
    hipError_t e = hipMemcpyAsync(counts_out, counts, bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream);
    if ((rc = check_launch(e, who))) return rc;
  }
  return AA_OK;
}

int aa_anchor_attn_fwd(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                       const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                       const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                       void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn,
                       void* workspace, size_t workspace_bytes, int32_t* counts_out,
                       int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                       int block_size, int step, double sm_scale, float theta_log2, int scale_mode, int geometry,
                       int dtype, void* stream) {
  return anchor_attn_impl("aa_anchor_attn_fwd", q, q_sb, q_sh, q_sn, k, k_sb, k_sh, k_sn, v, v_sb, v_sh, v_sn, out, o_sb, o_sh, o_sn,
                          workspace, workspace_bytes, counts_out, nullptr, nullptr, 1.0, batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size,
                          step, sm_scale, theta_log2, scale_mode, geometry, dtype, stream);
}

int aa_anchor_attn_ratio_fwd(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                             const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                             const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                             void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn,
                             void* workspace, size_t workspace_bytes, float* ratio, float* ratio_host, double denominator,
                             int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                             int block_size, int step, double sm_scale, float theta_log2, int scale_mode, int geometry,
                             int dtype, void* stream) {
  const char* who = "aa_anchor_attn_ratio_fwd";
  if (ratio == nullptr || !(denominator > 0.0)) {
    set_error("%s: ratio must not be NULL and denominator (%g) must be positive", who, denominator);
    return AA_EBADARG;
  }
  return anchor_attn_impl(who, q, q_sb, q_sh, q_sn, k, k_sb, k_sh, k_sn, v, v_sb, v_sh, v_sn, out, o_sb, o_sh, o_sn, workspace, workspace_bytes,
                          nullptr, ratio, ratio_host, denominator, batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step, sm_scale, theta_log2,
                          scale_mode, geometry, dtype, stream);
}

int aa_wait_ratio(const float* ratio_host, float unset, int timeout_us) {
  const volatile float* word = ratio_host;
  const auto end = std::chrono::steady_clock::now() + std::chrono::microseconds(timeout_us);
  for (;;) {
    for (int i = 0; i < 32; ++i) {
      if (*word != unset) return 1;
      __builtin_ia32_pause();
    }
    if (std::chrono::steady_clock::now() >= end) return *word != unset;
  }
}

int aa_sparsity_ratio(const int32_t* counts, int64_t n, double denominator, float* ratio, void* stream) {
  const char* who = "aa_sparsity_ratio";
  if (counts == nullptr || ratio == nullptr || n <= 0 || !(denominator > 0.0)) {
    set_error("%s: counts and ratio must not be NULL, n (%lld) and denominator (%g) must be positive", who, (long long)n, denominator);
    return AA_EBADARG;
  }
  return check_launch(launch_ratio(counts, n, 1.f / (float)denominator, ratio, (hipStream_t)stream), who);
}

int aa_dense_causal_fwd(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                        const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                        const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                        void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn,
                        int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                        float sm_scale, int dtype, void* stream) {
  const char* who = "aa_dense_causal_fwd";
  int rc;
  if ((rc = check_dtype(dtype, who))) return rc;
  if ((rc = check_common_dims({batch, n_q_heads, n_kv_heads, n_ctx, head_dim, 128, 16}, who))) return rc;
  if ((rc = check_tensor(q, q_sb, q_sh, q_sn, n_ctx, head_dim, who, "q"))) return rc;
  if ((rc = check_tensor(k, k_sb, k_sh, k_sn, n_ctx, head_dim, who, "k"))) return rc;
  if ((rc = check_tensor(v, v_sb, v_sh, v_sn, n_ctx, head_dim, who, "v"))) return rc;
  if ((rc = check_tensor(out, o_sb, o_sh, o_sn, n_ctx, head_dim, who, "out"))) return rc;
  FlashArgs a = {};
  a.q = (const uint16_t*)q; a.q_sb = q_sb; a.q_sh = q_sh; a.q_sn = q_sn;
  a.k = (const uint16_t*)k; a.k_sb = k_sb; a.k_sh = k_sh; a.k_sn = k_sn;
  a.v = (const uint16_t*)v; a.v_sb = v_sb; a.v_sh = v_sh; a.v_sn = v_sn;
  a.out = (uint16_t*)out; a.o_sb = o_sb; a.o_sh = o_sh; a.o_sn = o_sn;
  a.batch = batch; a.n_q_heads = n_q_heads; a.n_kv_heads = n_kv_heads; a.n_ctx = n_ctx; a.head_dim = head_dim;
  a.big_block = n_ctx; a.block_size = 128;  // one "big block": bb is always 0
  a.sm_scale = sm_scale; a.scale_mode = AA_SCALE_FP32; a.dtype = dtype;
  return check_launch(run_flash(a, 2, (hipStream_t)stream), who);
}

// Sizes of a rows-mode problem, checked and planned for its type; `masked`: with a boolean mask in the place of the causal rule.
static int plan_dense_rows(const char* who, FlashArgs& a, int batch, int n_q_heads, int n_kv_heads, int n_rows, int n_keys, int head_dim,
                           int causal_offset, bool masked, int dtype) {
  if (batch <= 0 || n_q_heads <= 0 || n_kv_heads <= 0 || n_rows <= 0 || n_keys <= 0 || causal_offset < 0) {
    set_error("%s: batch, head counts, n_rows and n_keys must be positive and causal_offset not negative (got %d, %d, %d, %d, %d, %d)", who,
              batch, n_q_heads, n_kv_heads, n_rows, n_keys, causal_offset);
    return AA_EBADARG;
  }
  if (n_q_heads % n_kv_heads != 0) {
    set_error("%s: n_kv_heads (%d) must divide n_q_heads (%d)", who, n_kv_heads, n_q_heads);
    return AA_EBADARG;
  }
  if (head_dim != 128 && head_dim != 64) {
    set_error("%s: head_dim %d is not supported (128 or 64)", who, head_dim);
    return AA_EUNSUPPORTED;
  }
  if (n_keys > (1 << 20) || n_rows > (1 << 20) || causal_offset > (1 << 20)) {
    set_error("%s: %d rows, %d keys or causal offset %d is more than 2^20", who, n_rows, n_keys, causal_offset);
    return AA_EUNSUPPORTED;
  }
  const int64_t col_blocks = ((int64_t)n_rows * (n_q_heads / n_kv_heads) + 127) / 128;
  // (the mask kernel counts column blocks and batch in its grid's y and z, and a row's packed mask has a 32-bit byte offset)
  const int64_t blocks = (int64_t)batch * n_kv_heads * col_blocks;
  if (blocks > 0xffffff || (masked && (col_blocks > 65535 || batch > 65535 || (int64_t)n_rows * ((n_keys + 63) / 64) * 8 > 0xffffffffLL))) {
    set_error("%s: problem too large for one launch", who);
    return AA_EUNSUPPORTED;
  }
  a.batch = batch; a.n_q_heads = n_q_heads; a.n_kv_heads = n_kv_heads; a.n_rows = n_rows; a.n_ctx = n_keys; a.head_dim = head_dim; a.dtype = dtype;
  a.causal_offset = masked ? n_keys : causal_offset;
  a.mask_words_per_row = masked ? (n_keys + 63) / 64 : 0;
  a.big_block = n_keys; a.block_size = 128;  // (unused in this mode; not zero)
  if (decode_takes(n_rows, n_q_heads / n_kv_heads, masked)) {
    a.mask_words_per_row = 0;  // (the decode kernel reads the byte mask itself)
    plan_decode(a);
  } else {
    plan_rows(a);
  }
  // (a launch takes less than 2^32 threads, 256 to a column block and chunk)
  if (blocks * a.n_chunks > 0xffffff) {
    set_error("%s: problem too large for one launch", who);
    return AA_EUNSUPPORTED;
  }
  return AA_OK;
}

// Scratch of a rows-mode problem: the state of its chunks, then the packed mask and its tile flags.
struct RowsScratch {
  int64_t state_columns;
  size_t words, flags, total;
};
static RowsScratch carve_rows(const FlashArgs& a, bool decode) {
  RowsScratch r;
  const int columns = decode ? a.n_rows * (a.n_q_heads / a.n_kv_heads) : 128 * a.n_col_blocks;
  r.state_columns = a.n_chunks > 1 ? (int64_t)a.batch * a.n_kv_heads * a.n_chunks * columns : 0;
  r.words = align256((size_t)r.state_columns * (a.head_dim + 2) * 4);  // accumulators, maxima, sums
  r.flags = r.words + align256((size_t)a.batch * a.n_rows * a.mask_words_per_row * 8);
  r.total = r.flags + (size_t)a.batch * a.n_col_blocks * a.mask_words_per_row;
  return r;
}

size_t aa_dense_rows_workspace_bytes_of(int batch, int n_q_heads, int n_kv_heads, int n_rows, int n_keys, int head_dim, int causal_offset,
                                        int masked, int dtype) {
  const char* who = "aa_dense_rows_workspace_bytes_of";
  FlashArgs a = {};
  if (check_dtype(dtype, who) ||
      plan_dense_rows(who, a, batch, n_q_heads, n_kv_heads, n_rows, n_keys, head_dim, causal_offset, masked != 0, dtype))
    return 0;
  return carve_rows(a, decode_takes(n_rows, n_q_heads / n_kv_heads, masked != 0)).total;
}

size_t aa_dense_rows_workspace_bytes(int batch, int n_q_heads, int n_kv_heads, int n_rows, int n_keys, int head_dim, int causal_offset,
                                     int masked) {
  const char* who = "aa_dense_rows_workspace_bytes";
  size_t most = 0;
  for (const int dtype : {AA_DTYPE_BF16, AA_DTYPE_F16}) {
    FlashArgs a = {};
    if (plan_dense_rows(who, a, batch, n_q_heads, n_kv_heads, n_rows, n_keys, head_dim, causal_offset, masked != 0, dtype)) return 0;
    most = std::max(most, carve_rows(a, decode_takes(n_rows, n_q_heads / n_kv_heads, masked != 0)).total);
  }
  return most;
}

// Tensors and scratch of a planned rows-mode problem, checked and put into `a`.
static int rows_args(const char* who, FlashArgs& a, const RowsScratch& r, const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                     const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                     void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn, void* workspace, size_t workspace_bytes, float sm_scale, int dtype) {
  int rc;
  if ((rc = check_tensor(q, q_sb, q_sh, q_sn, a.n_rows, a.head_dim, who, "q"))) return rc;
  if ((rc = check_tensor(k, k_sb, k_sh, k_sn, a.n_ctx, a.head_dim, who, "k"))) return rc;
  if ((rc = check_tensor(v, v_sb, v_sh, v_sn, a.n_ctx, a.head_dim, who, "v"))) return rc;
  if ((rc = check_tensor(out, o_sb, o_sh, o_sn, a.n_rows, a.head_dim, who, "out"))) return rc;
  if (!(sm_scale > 0.f)) {  // the running maxima are those of the raw dot products
    set_error("%s: sm_scale %g must be positive", who, (double)sm_scale);
    return AA_EUNSUPPORTED;
  }
  if (r.total > 0) {
    if ((rc = check_ptr(workspace, who, "workspace"))) return rc;
    if (workspace_bytes < r.total) {
      set_error("%s: workspace has %zu bytes, %zu needed", who, workspace_bytes, r.total);
      return AA_EBADARG;
    }
  }
  a.q = (const uint16_t*)q; a.q_sb = q_sb; a.q_sh = q_sh; a.q_sn = q_sn;
  a.k = (const uint16_t*)k; a.k_sb = k_sb; a.k_sh = k_sh; a.k_sn = k_sn;
  a.v = (const uint16_t*)v; a.v_sb = v_sb; a.v_sh = v_sh; a.v_sn = v_sn;
  a.out = (uint16_t*)out; a.o_sb = o_sb; a.o_sh = o_sh; a.o_sn = o_sn;
  a.acc_out = (float*)workspace; a.M_out = a.acc_out + r.state_columns * a.head_dim; a.L_out = a.M_out + r.state_columns;
  a.acc_frag = a.acc_out; a.M = a.M_out; a.L = a.L_out;
  a.sm_scale = sm_scale; a.scale_mode = AA_SCALE_FP32; a.dtype = dtype;
  return AA_OK;
}

int aa_dense_rows_fwd(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                      const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                      const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                      void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn,
                      const uint8_t* mask, int64_t mask_sb, int64_t mask_sn,
                      void* workspace, size_t workspace_bytes,
                      int batch, int n_q_heads, int n_kv_heads, int n_rows, int n_keys, int head_dim, int causal_offset,
                      float sm_scale, int dtype, void* stream) {
  const char* who = "aa_dense_rows_fwd";
  FlashArgs a = {};
  int rc;
  if ((rc = check_dtype(dtype, who))) return rc;
  if ((rc = plan_dense_rows(who, a, batch, n_q_heads, n_kv_heads, n_rows, n_keys, head_dim, causal_offset, mask != nullptr, dtype)))
    return rc;
  const bool decode = decode_takes(n_rows, n_q_heads / n_kv_heads, mask != nullptr);
  const RowsScratch r = carve_rows(a, decode);
  if ((rc = rows_args(who, a, r, q, q_sb, q_sh, q_sn, k, k_sb, k_sh, k_sn, v, v_sb, v_sh, v_sn, out, o_sb, o_sh, o_sn, workspace, workspace_bytes,
                      sm_scale, dtype)))
    return rc;
  if (decode) {
    a.mask_bytes = mask; a.mask_sb = mask_sb;
    return check_launch(launch_decode(a, (hipStream_t)stream), who);
  }
  if (mask != nullptr) {
    char* ws = static_cast<char*>(workspace);
    a.mask_words = (const uint64_t*)(ws + r.words);
    a.tile_flags = (const uint8_t*)(ws + r.flags);
    if ((rc = check_launch(launch_mask_pack(a, mask, mask_sb, mask_sn, (hipStream_t)stream), who))) return rc;
  }
  if ((rc = check_launch(run_flash(a, mask != nullptr ? 4 : 3, (hipStream_t)stream), who))) return rc;
  return a.n_chunks > 1 ? check_launch(launch_rows_combine(a, (hipStream_t)stream), who) : AA_OK;
}

// A rows-mode problem beside the operator, planned.
struct RowsBeside {
  bool shares;  // stage 1's launch (else it has its own after the operator: a few rows are the decode kernel's)
  FlashArgs args;
  RowsScratch scratch;
  size_t operator_bytes;  // the operator's scratch; the rows' follows it
};
static int plan_beside(const char* who, RowsBeside& r, int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim, int block_size, int step,
                       int n_rows, int n_keys, int causal_offset, int dtype) {
  const Dims dims = {batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step};
  int rc;
  r.args = FlashArgs{};
  if ((rc = check_dims(dims, who)) || 
      (rc = plan_dense_rows(who, r.args, batch, n_q_heads, n_kv_heads, n_rows, n_keys, head_dim, causal_offset, false, dtype)))
    return rc;
  const bool decode = decode_takes(n_rows, n_q_heads / n_kv_heads, false);
  r.shares = false;
  if (!decode) {
    FlashArgs beside = r.args, anchor = {};
    anchor.batch = batch; anchor.n_q_heads = n_q_heads; anchor.n_ctx = n_ctx; anchor.head_dim = head_dim; anchor.big_block = block_size * step;
    plan_rows_beside(beside, anchor);
    // (a launch takes less than 2^32 threads, 256 to a work-group)
    r.shares = (int64_t)batch * n_q_heads * (n_ctx / 128) + (int64_t)batch * n_kv_heads * beside.n_col_blocks * beside.n_chunks + 8 <= 0xffffff;
    if (r.shares) r.args = beside;
  }
  r.scratch = carve_rows(r.args, decode);
  r.operator_bytes = carve(batch, n_q_heads, n_ctx, head_dim, block_size, step).total;
  return AA_OK;
}

size_t aa_anchor_attn_rows_workspace_bytes(int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim, int block_size, int step,
                                           int n_rows, int n_keys, int causal_offset) {
  const char* who = "aa_anchor_attn_rows_workspace_bytes";
  size_t most = 0;
  for (const int dtype : {AA_DTYPE_BF16, AA_DTYPE_F16}) {
    RowsBeside r;
    if (plan_beside(who, r, batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step, n_rows, n_keys, causal_offset, dtype)) return 0;
    most = std::max(most, r.operator_bytes + r.scratch.total);
    if (r.shares) break;  // (then the type does not matter)
  }
  return most;
}

int aa_anchor_attn_rows_fwd(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn,
                            const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                            const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sn,
                            void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn,
                            const void* rq, int64_t rq_sb, int64_t rq_sh, int64_t rq_sn,
                            const void* rk, int64_t rk_sb, int64_t rk_sh, int64_t rk_sn,
                            const void* rv, int64_t rv_sb, int64_t rv_sh, int64_t rv_sn,
                            void* rout, int64_t ro_sb, int64_t ro_sh, int64_t ro_sn, int n_rows, int n_keys, int causal_offset, float rows_scale,
                            void* workspace, size_t workspace_bytes, int32_t* counts_out, float* ratio, float* ratio_host, double denominator,
                            int batch, int n_q_heads, int n_kv_heads, int n_ctx, int head_dim,
                            int block_size, int step, double sm_scale, float theta_log2, int scale_mode, int geometry,
                            int dtype, void* stream) {
  const char* who = "aa_anchor_attn_rows_fwd";
  RowsBeside r;
  int rc;
  if ((rc = check_dtype(dtype, who))) return rc;
  if ((rc = plan_beside(who, r, batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step, n_rows, n_keys, causal_offset, dtype))) return rc;
  if ((rc = check_ptr(workspace, who, "workspace"))) return rc;
  if (workspace_bytes < r.operator_bytes + r.scratch.total) {
    set_error("%s: workspace has %zu bytes, %zu needed", who, workspace_bytes, r.operator_bytes + r.scratch.total);
    return AA_EBADARG;
  }
  if (ratio != nullptr && !(denominator > 0.0)) {
    set_error("%s: denominator (%g) must be positive", who, denominator);
    return AA_EBADARG;
  }
  char* rows_ws = static_cast<char*>(workspace) + r.operator_bytes;
  if ((rc = rows_args(who, r.args, r.scratch, rq, rq_sb, rq_sh, rq_sn, rk, rk_sb, rk_sh, rk_sn, rv, rv_sb, rv_sh, rv_sn, rout, ro_sb, ro_sh, ro_sn,
                      rows_ws, r.scratch.total, rows_scale, dtype)))
    return rc;
  if ((rc = anchor_attn_impl(who, q, q_sb, q_sh, q_sn, k, k_sb, k_sh, k_sn, v, v_sb, v_sh, v_sn, out, o_sb, o_sh, o_sn, workspace, r.operator_bytes,
                             counts_out, ratio, ratio_host, denominator, batch, n_q_heads, n_kv_heads, n_ctx, head_dim, block_size, step, sm_scale,
                             theta_log2, scale_mode, geometry, dtype, stream, r.shares ? &r.args : nullptr)))
    return rc;
  if (r.shares) return AA_OK;
  return aa_dense_rows_fwd(rq, rq_sb, rq_sh, rq_sn, rk, rk_sb, rk_sh, rk_sn, rv, rv_sb, rv_sh, rv_sn, rout, ro_sb, ro_sh, ro_sn, nullptr, 0, 0, rows_ws,
                           r.scratch.total, batch, n_q_heads, n_kv_heads, n_rows, n_keys, head_dim, causal_offset, rows_scale, dtype, stream);
}

int aa_rms_norm(const void* x, const void* weight, void* out, int64_t rows, int hidden, float eps, int dtype, void* stream) {
  const char* who = "aa_rms_norm";
  int rc;
  if ((rc = check_dtype(dtype, who)) || (rc = check_ptr(x, who, "x")) || (rc = check_ptr(weight, who, "weight")) || (rc = check_ptr(out, who, "out"))) return rc;
  if (rows <= 0 || rows > 0xffffff || hidden <= 0 || hidden > 16384 || hidden % 8 != 0) {  // (a launch takes less than 2^32 threads, 256 a row)
    set_error("%s: %lld rows of %d elements are not supported (at most 2^24 - 1 rows of at most 16384, a multiple of 8)", who, (long long)rows, hidden);
    return AA_EUNSUPPORTED;
  }
  return check_launch(launch_rms_norm((const uint16_t*)x, (const uint16_t*)weight, (uint16_t*)out, rows, hidden, eps, dtype, (hipStream_t)stream), who);
}

int aa_silu_mul(const void* gate, const void* up, void* out, int64_t n, int dtype, void* stream) {
  const char* who = "aa_silu_mul";
  int rc;
  if ((rc = check_dtype(dtype, who)) || (rc = check_ptr(gate, who, "gate")) || (rc = check_ptr(up, who, "up")) || (rc = check_ptr(out, who, "out"))) return rc;
  if (n <= 0 || n % 8 != 0 || n / 8 > 0xffffff00LL) {
    set_error("%s: %lld elements are not supported (a multiple of 8, at most 2^35)", who, (long long)n);
    return AA_EUNSUPPORTED;
  }
  return check_launch(launch_silu_mul((const uint16_t*)gate, (const uint16_t*)up, (uint16_t*)out, n, dtype, (hipStream_t)stream), who);
}

int aa_rope(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_sn, const void* k, int64_t k_sb, int64_t k_sh, int64_t k_sn,
            void* q_out, int64_t qo_sb, int64_t qo_sh, int64_t qo_sn, void* k_out, int64_t ko_sb, int64_t ko_sh, int64_t ko_sn,
            const void* cos, const void* sin, int64_t cs_sb, int batch, int n_q_heads, int n_kv_heads, int n_tokens, int head_dim,
            int dtype, void* stream) {
  const char* who = "aa_rope";
  int rc;
  if (batch <= 0 || n_q_heads <= 0 || n_kv_heads <= 0 || n_tokens <= 0) {
    set_error("%s: batch, head counts and n_tokens must be positive (got %d, %d, %d, %d)", who, batch, n_q_heads, n_kv_heads, n_tokens);
    return AA_EBADARG;
  }
  if (head_dim <= 0 || head_dim > 1024 || head_dim % 16 != 0 ||
      ((int64_t)n_q_heads + n_kv_heads + 3) / 4 * (head_dim / 16) >= 0xffffff00LL / batch / n_tokens) {
    set_error("%s: %d x %d tokens of %d + %d heads of %d are not supported (a multiple of 16 up to 1024, fewer than 2^32 pieces of 64 elements)", who,
              batch, n_tokens, n_q_heads, n_kv_heads, head_dim);
    return AA_EUNSUPPORTED;
  }
  if ((rc = check_dtype(dtype, who)) || (rc = check_tensor(q, q_sb, q_sh, q_sn, n_tokens, head_dim, who, "q")) ||
      (rc = check_tensor(k, k_sb, k_sh, k_sn, n_tokens, head_dim, who, "k")) || (rc = check_tensor(q_out, qo_sb, qo_sh, qo_sn, n_tokens, head_dim, who, "q_out")) ||
      (rc = check_tensor(k_out, ko_sb, ko_sh, ko_sn, n_tokens, head_dim, who, "k_out")) || (rc = check_ptr(cos, who, "cos")) || (rc = check_ptr(sin, who, "sin")))
    return rc;
  if (cs_sb % 8 != 0) {
    set_error("%s: cos and sin must have a batch stride that is a multiple of 8 elements (got %lld)", who, (long long)cs_sb);
    return AA_EMISALIGNED;
  }
  RopeArgs a = {(const uint16_t*)q, q_sb, q_sh, q_sn, (const uint16_t*)k, k_sb, k_sh, k_sn, (uint16_t*)q_out, qo_sb, qo_sh, qo_sn,
                (uint16_t*)k_out, ko_sb, ko_sh, ko_sn, (const uint16_t*)cos, (const uint16_t*)sin, cs_sb, batch, n_q_heads, n_kv_heads, n_tokens, head_dim};
  return check_launch(launch_rope(a, dtype, (hipStream_t)stream), who);
}

}  // extern "C"
