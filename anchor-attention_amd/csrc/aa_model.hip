// The passes between a patched model's matrix products on gfx950: root-mean-square normalisation, the gated activation of the MLP and the
// rotary position embedding.
//
// All are bound by reading and writing each element once.  The framework forms them of single operations, each a pass over memory
// with float32 intermediates: eight for a norm (6001 x 2048 bf16: 91 us; 49 MB at the rate of a large copy are 10), two for the
// activation and product (6001 x 8192: 83 us; 295 MB, 63), ten for the embedding (6001 tokens, 32/8 heads of 64: 135 us; 61 MB, 13).  The arithmetic and the 16-bit roundings between the operations are theirs;
// only the order of the sum of squares differs.
#include "aa_common.h"
#include "aa_kernels.h"

namespace aa {

// One work-group per row, which stays in registers between the sum of squares and the scaling: ITS pieces of 256 x 8 elements.
template <typename T, int ITS>
__global__ void __launch_bounds__(256) rms_norm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ weight, uint16_t* __restrict__ out,
                                                       const int hidden, const float eps) {
  __shared__ float part[4];
  const int64_t row = (int64_t)blockIdx.x * hidden;
  uint4 raw[ITS];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < ITS; ++i) {
    const int at = (256 * i + threadIdx.x) * 8;
    raw[i] = uint4{0u, 0u, 0u, 0u};
    if (at < hidden) raw[i] = *reinterpret_cast<const uint4*>(x + row + at);
  }
#pragma unroll
  for (int i = 0; i < ITS; ++i) {
    const uint32_t w[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) sum += T::lo(w[j]) * T::lo(w[j]) + T::hi(w[j]) * T::hi(w[j]);
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum;
  __syncthreads();
  const float scale = rsqrtf(((part[0] + part[1]) + (part[2] + part[3])) * (1.f / (float)hidden) + eps);
#pragma unroll
  for (int i = 0; i < ITS; ++i) {
    const int at = (256 * i + threadIdx.x) * 8;
    if (at >= hidden) continue;
    const uint4 wt = *reinterpret_cast<const uint4*>(weight + at);
    const uint32_t w[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w}, g[4] = {wt.x, wt.y, wt.z, wt.w};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t y = T::pack(T::lo(w[j]) * scale, T::hi(w[j]) * scale);  // rounded before it meets the weight
      o[j] = T::pack(T::lo(g[j]) * T::lo(y), T::hi(g[j]) * T::hi(y));
    }
    *reinterpret_cast<uint4*>(out + row + at) = uint4{o[0], o[1], o[2], o[3]};
  }
}

template <typename T>
static hipError_t launch_rms_norm_for(const uint16_t* x, const uint16_t* weight, uint16_t* out, int64_t rows, int hidden, float eps, hipStream_t stream) {
  const dim3 grid((uint32_t)rows), block(256);
  if (hidden <= 2048) hipLaunchKernelGGL((rms_norm_kernel<T, 1>), grid, block, 0, stream, x, weight, out, hidden, eps);
  else if (hidden <= 4096) hipLaunchKernelGGL((rms_norm_kernel<T, 2>), grid, block, 0, stream, x, weight, out, hidden, eps);
  else if (hidden <= 8192) hipLaunchKernelGGL((rms_norm_kernel<T, 4>), grid, block, 0, stream, x, weight, out, hidden, eps);
  else hipLaunchKernelGGL((rms_norm_kernel<T, 8>), grid, block, 0, stream, x, weight, out, hidden, eps);  // up to 16384
  return hipGetLastError();
}

hipError_t launch_rms_norm(const uint16_t* x, const uint16_t* weight, uint16_t* out, int64_t rows, int hidden, float eps, int dtype, hipStream_t stream) {
  return dtype == 0 ? launch_rms_norm_for<Bf16>(x, weight, out, rows, hidden, eps, stream)
                    : launch_rms_norm_for<F16>(x, weight, out, rows, hidden, eps, stream);
}

// out = round16(silu(gate)) * up, eight elements a thread.
template <typename T>
__global__ void __launch_bounds__(256) silu_mul_kernel(const uint16_t* __restrict__ gate, const uint16_t* __restrict__ up, uint16_t* __restrict__ out,
                                                       const int64_t pieces) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= pieces) return;
  const uint4 a = reinterpret_cast<const uint4*>(gate)[i], b = reinterpret_cast<const uint4*>(up)[i];
  const uint32_t g[4] = {a.x, a.y, a.z, a.w}, u[4] = {b.x, b.y, b.z, b.w};
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float g0 = T::lo(g[j]), g1 = T::hi(g[j]);
    const uint32_t s = T::pack(g0 / (1.f + expf(-g0)), g1 / (1.f + expf(-g1)));
    o[j] = T::pack(T::lo(s) * T::lo(u[j]), T::hi(s) * T::hi(u[j]));
  }
  reinterpret_cast<uint4*>(out)[i] = uint4{o[0], o[1], o[2], o[3]};
}

hipError_t launch_silu_mul(const uint16_t* gate, const uint16_t* up, uint16_t* out, int64_t n, int dtype, hipStream_t stream) {
  const dim3 grid((uint32_t)((n / 8 + 255) / 256)), block(256);
  if (dtype == 0) hipLaunchKernelGGL(silu_mul_kernel<Bf16>, grid, block, 0, stream, gate, up, out, n / 8);
  else hipLaunchKernelGGL(silu_mul_kernel<F16>, grid, block, 0, stream, gate, up, out, n / 8);
  return hipGetLastError();
}

// x * cos + rotate(x) * sin, where rotate takes (first, second half of a head) to (-second, first): each product and the sum rounded, as
// the single operations do.  A thread takes eight elements of both halves of up to four heads of a token, of queries and keys alike, which share
// its cosines and sines.  6001 tokens, 32/8 heads of 64: 14 us.
template <typename T>
__global__ void __launch_bounds__(256) rope_kernel(const RopeArgs p) {
  const uint32_t pieces = (uint32_t)p.head_dim / 16u, heads = (uint32_t)(p.n_q_heads + p.n_kv_heads), groups = (heads + 3u) / 4u;
  uint32_t id = blockIdx.x * 256u + threadIdx.x;
  const uint32_t piece = id % pieces;  id /= pieces;
  const uint32_t first = id % groups;  id /= groups;
  const uint32_t n = id % (uint32_t)p.n_tokens, b = id / (uint32_t)p.n_tokens;
  if (b >= (uint32_t)p.batch) return;
  const int half = p.head_dim / 2;
  const int64_t at = (int64_t)b * p.cs_sb + (int64_t)n * p.head_dim + 8 * piece;
  const uint4 cl = *reinterpret_cast<const uint4*>(p.cos + at), ch = *reinterpret_cast<const uint4*>(p.cos + at + half);
  const uint4 sl = *reinterpret_cast<const uint4*>(p.sin + at), sh = *reinterpret_cast<const uint4*>(p.sin + at + half);
  const uint32_t c0[4] = {cl.x, cl.y, cl.z, cl.w}, c1[4] = {ch.x, ch.y, ch.z, ch.w};
  const uint32_t s0[4] = {sl.x, sl.y, sl.z, sl.w}, s1[4] = {sh.x, sh.y, sh.z, sh.w};
  uint4 lo[4], hi[4];
  uint16_t* to[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t h = first + j * groups;
    const bool is_q = h < (uint32_t)p.n_q_heads;
    const int64_t hh = is_q ? h : h - (uint32_t)p.n_q_heads;
    to[j] = nullptr;
    if (h >= heads) continue;
    const uint16_t* from = (is_q ? p.q + b * p.q_sb + hh * p.q_sh + n * p.q_sn : p.k + b * p.k_sb + hh * p.k_sh + n * p.k_sn) + 8 * piece;
    to[j] = (is_q ? p.q_out + b * p.qo_sb + hh * p.qo_sh + n * p.qo_sn : p.k_out + b * p.ko_sb + hh * p.ko_sh + n * p.ko_sn) + 8 * piece;
    lo[j] = *reinterpret_cast<const uint4*>(from);
    hi[j] = *reinterpret_cast<const uint4*>(from + half);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (to[j] == nullptr) continue;
    const uint32_t x0[4] = {lo[j].x, lo[j].y, lo[j].z, lo[j].w}, x1[4] = {hi[j].x, hi[j].y, hi[j].z, hi[j].w};
    uint32_t y0[4], y1[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t a = T::pack(T::lo(x0[i]) * T::lo(c0[i]), T::hi(x0[i]) * T::hi(c0[i])), b_ = T::pack(-T::lo(x1[i]) * T::lo(s0[i]), -T::hi(x1[i]) * T::hi(s0[i]));
      const uint32_t c = T::pack(T::lo(x1[i]) * T::lo(c1[i]), T::hi(x1[i]) * T::hi(c1[i])), d = T::pack(T::lo(x0[i]) * T::lo(s1[i]), T::hi(x0[i]) * T::hi(s1[i]));
      y0[i] = T::pack(T::lo(a) + T::lo(b_), T::hi(a) + T::hi(b_));
      y1[i] = T::pack(T::lo(c) + T::lo(d), T::hi(c) + T::hi(d));
    }
    *reinterpret_cast<uint4*>(to[j]) = uint4{y0[0], y0[1], y0[2], y0[3]};
    *reinterpret_cast<uint4*>(to[j] + half) = uint4{y1[0], y1[1], y1[2], y1[3]};
  }
}

hipError_t launch_rope(const RopeArgs& a, int dtype, hipStream_t stream) {
  const int64_t threads = (int64_t)a.batch * a.n_tokens * ((a.n_q_heads + a.n_kv_heads + 3) / 4) * (a.head_dim / 16);
  const dim3 grid((uint32_t)((threads + 255) / 256)), block(256);
  if (dtype == 0) hipLaunchKernelGGL(rope_kernel<Bf16>, grid, block, 0, stream, a);
  else hipLaunchKernelGGL(rope_kernel<F16>, grid, block, 0, stream, a);
  return hipGetLastError();
}

}  // namespace aa
