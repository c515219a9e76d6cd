// Projections and rotary embedding of an attention layer: what surrounds the prefill and decode kernels in the
// reference's Llama forward (xattn/src/load_llama.py:119-150, 207-218).
//
//  qkv_rope_gemv_kernel / gemv: y = W x for ONE token.  Bound by HBM: every weight is read once and used once, 84 MB
//    for a 4096-wide layer with 32 + 2 * 8 heads.  A wavefront takes four weight rows at a time (for q and k two
//    rotary pairs d, d + 64 and their neighbours, so that the rotation happens in registers), every load is a full
//    1 KiB of one row, and 20 of them are in flight per wavefront before the first is used.  The library GEMM with
//    one row left most of the chip idle: 47 us for the four products of that layer (1.8 TB/s), and the rotation
//    another 13 launches.  (Loaded "not temporal" the weights come 4 to 8 % faster from memory, but a layer whose weights are in the
//    memory-side cache still is 1 to 3 % slower.)  proj_gemm.hip has the products of more tokens.
//  rope_kernel: the rotation of q and k of many tokens in place, one read and one write of both.  The reference's
//    expression is ten elementwise kernels over them.
//
// Both round where the reference's bf16 tensor expression q * cos + rotate_half(q) * sin rounds: after the projection,
// after each product and after the sum.
#include "rotate.h"
#include "xattn_hip.h"

namespace xattn {

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

struct GemvParams {
  const __bf16* x;
  const __bf16* w[3];        // weights, rows of K contiguous elements
  const __bf16* bias[3];     // or null
  __bf16* y[3];
  int64_t w_sn[3];           // row stride, elements
  int units[3];              // four-row units of each product
  int K;
  const __bf16* cos;         // 128 each; null: no rotation
  const __bf16* sin;
};

constexpr int kGemvBatch = 4;    // 512-element chunks of a row per batch of loads

// kRope: a unit is rows d, d+1, d+64, d+65 of one head (products 0 and 1 rotated, 2 not); otherwise four rows in order
template <bool kRope>
__global__ __launch_bounds__(256) void gemv_kernel(GemvParams p) {
  const int lane = threadIdx.x & 63;
  int unit = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  int t = 0;
  if (kRope) {
    if (unit >= p.units[0]) { unit -= p.units[0]; t = 1; }
    if (t == 1 && unit >= p.units[1]) { unit -= p.units[1]; t = 2; }
  }
  if (unit >= p.units[t]) return;
  int row[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    row[i] = kRope ? (unit >> 5) * 128 + (unit & 31) * 2 + (i & 1) + (i >> 1) * 64 : unit * 4 + i;
  // loads past the end of a row return zeros
  __amdgpu_buffer_rsrc_t wres[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    wres[i] = __builtin_amdgcn_make_buffer_rsrc((void*)(p.w[t] + (int64_t)row[i] * p.w_sn[t]), 0, p.K * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, p.K * 2, 0x00020000);

  u32x4 wv[2][kGemvBatch][4], xv[2][kGemvBatch];
  auto load = [&](int b, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < kGemvBatch; ++c) {
      const int off = ((b * kGemvBatch + c) * 64 + lane) * 16;
      xv[buf][c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xres, off, 0, 0));
#pragma unroll
      for (int i = 0; i < 4; ++i)
        wv[buf][c][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wres[i], off, 0, 0));
    }
  };
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  auto use = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < kGemvBatch; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[i] = __builtin_fmaf(bf16_lo(wv[buf][c][i][e]), bf16_lo(xv[buf][c][e]), acc[i]);
          acc[i] = __builtin_fmaf(bf16_hi(wv[buf][c][i][e]), bf16_hi(xv[buf][c][e]), acc[i]);
        }
  };
  const int batches = (p.K + kGemvBatch * 512 - 1) / (kGemvBatch * 512);
  load(0, 0);
  for (int b = 0; b < batches; b += 2) {
    load(b + 1, 1);
    __builtin_amdgcn_sched_barrier(0);
    use(0);
    if (b + 2 < batches) load(b + 2, 0);
    __builtin_amdgcn_sched_barrier(0);
    use(1);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) acc[i] += __shfl_xor(acc[i], d, 64);
  if (lane == 0) {
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = bf16_round(acc[i] + (p.bias[t] ? (float)p.bias[t][row[i]] : 0.f));
    if (kRope && t < 2) {
      const int d = (unit & 31) * 2;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        rotate_pair(y[i], y[i + 2], (float)p.cos[d + i], (float)p.cos[d + i + 64], (float)p.sin[d + i], (float)p.sin[d + i + 64]);
    }
    *reinterpret_cast<uint32_t*>(p.y[t] + row[0]) = pack_bf16(y[0], y[1]);
    *reinterpret_cast<uint32_t*>(p.y[t] + row[2]) = pack_bf16(y[2], y[3]);
  }
}

struct RopeParams {
  __bf16* q;                 // [tokens][heads][128], rotated in place
  __bf16* k;
  const __bf16* cos;         // [tokens][128]
  const __bf16* sin;
  int64_t cos_sn, sin_sn;    // token stride, elements
  int heads, kv_heads;
  int64_t total;             // tokens * (heads + kv_heads) * 8 threads, one per 8 rotary pairs
};

__global__ __launch_bounds__(256) void rope_kernel(RopeParams p) {
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= p.total) return;
  const int c = (int)(id & 7);
  const uint32_t hd = (uint32_t)(id >> 3);                 // the host refuses 2^31 (token, head) pairs or more
  const uint32_t all = (uint32_t)(p.heads + p.kv_heads);
  const uint32_t tok = hd / all, h = hd - tok * all;
  __bf16* base = h < (uint32_t)p.heads ? p.q + ((int64_t)tok * p.heads + h) * kHeadDim
                                       : p.k + ((int64_t)tok * p.kv_heads + (h - p.heads)) * kHeadDim;
  base += c * 8;
  const __bf16* cs = p.cos + (int64_t)tok * p.cos_sn + c * 8;
  const __bf16* sn = p.sin + (int64_t)tok * p.sin_sn + c * 8;
  bf16x8 y0 = *reinterpret_cast<const bf16x8*>(base), y1 = *reinterpret_cast<const bf16x8*>(base + 64);
  rotate_chunks(y0, y1, cs, sn);
  *reinterpret_cast<bf16x8*>(base) = y0;
  *reinterpret_cast<bf16x8*>(base + 64) = y1;
}

}  // namespace xattn

using namespace xattn;

namespace {
bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool a4(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3) == 0; }
// a row's loads are 16 bytes at 32-bit offsets
bool width_ok(int K) { return K >= 8 && K % 8 == 0 && K <= (1 << 24); }
}  // namespace

extern "C" int xattn_qkv_rope_gemv(const void* x, int width, const void* wq, int64_t wq_stride, const void* bq,
                                   const void* wk, int64_t wk_stride, const void* bk, const void* wv, int64_t wv_stride,
                                   const void* bv, const void* cos, const void* sin, void* q, void* k, void* v,
                                   int num_heads, int num_kv_heads, int head_dim, void* stream) {
  if (!x || !wq || !wk || !wv || !cos || !sin || !q || !k || !v) return XATTN_ERR_NULL;
  if (head_dim != kHeadDim) return XATTN_ERR_HEAD_DIM;
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads > 4096 || num_kv_heads > 4096) return XATTN_ERR_HEADS;
  if (!width_ok(width) || wq_stride < width || wk_stride < width || wv_stride < width) return XATTN_ERR_SHAPE;
  if (wq_stride % 8 || wk_stride % 8 || wv_stride % 8) return XATTN_ERR_ALIGN;
  if (!a16(x) || !a16(wq) || !a16(wk) || !a16(wv) || !a4(q) || !a4(k) || !a4(v)) return XATTN_ERR_ALIGN;
  GemvParams p{};
  p.x = static_cast<const __bf16*>(x);
  const void *w[3] = {wq, wk, wv}, *b[3] = {bq, bk, bv};
  void* y[3] = {q, k, v};
  const int64_t sn[3] = {wq_stride, wk_stride, wv_stride};
  const int n[3] = {num_heads, num_kv_heads, num_kv_heads};
  int units = 0;
  for (int i = 0; i < 3; ++i) {
    p.w[i] = static_cast<const __bf16*>(w[i]);
    p.bias[i] = static_cast<const __bf16*>(b[i]);
    p.y[i] = static_cast<__bf16*>(y[i]);
    p.w_sn[i] = sn[i];
    units += p.units[i] = n[i] * 32;
  }
  p.K = width;
  p.cos = static_cast<const __bf16*>(cos);
  p.sin = static_cast<const __bf16*>(sin);
  hipLaunchKernelGGL(gemv_kernel<true>, dim3((unsigned)(units + 3) / 4), dim3(256), 0, static_cast<hipStream_t>(stream), p);
  return hipGetLastError() == hipSuccess ? XATTN_OK : XATTN_ERR_LAUNCH;
}

extern "C" int xattn_gemv(const void* x, int width, const void* w, int64_t w_stride, const void* bias, void* y, int rows,
                          void* stream) {
  if (!x || !w || !y) return XATTN_ERR_NULL;
  if (!width_ok(width) || w_stride < width || rows < 4 || rows % 4) return XATTN_ERR_SHAPE;
  if (w_stride % 8 || !a16(x) || !a16(w) || !a4(y)) return XATTN_ERR_ALIGN;
  GemvParams p{};
  p.x = static_cast<const __bf16*>(x);
  p.w[0] = static_cast<const __bf16*>(w);
  p.bias[0] = static_cast<const __bf16*>(bias);
  p.y[0] = static_cast<__bf16*>(y);
  p.w_sn[0] = w_stride;
  p.units[0] = rows / 4;
  p.K = width;
  hipLaunchKernelGGL(gemv_kernel<false>, dim3((unsigned)(p.units[0] + 3) / 4), dim3(256), 0, static_cast<hipStream_t>(stream), p);
  return hipGetLastError() == hipSuccess ? XATTN_OK : XATTN_ERR_LAUNCH;
}

extern "C" int xattn_rope(void* q, void* k, const void* cos, const void* sin, int64_t cos_stride, int64_t sin_stride,
                          int tokens, int num_heads, int num_kv_heads, int head_dim, void* stream) {
  if (!q || !k || !cos || !sin) return XATTN_ERR_NULL;
  if (head_dim != kHeadDim) return XATTN_ERR_HEAD_DIM;
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads > 4096 || num_kv_heads > 4096) return XATTN_ERR_HEADS;
  if (tokens <= 0 || cos_stride < 0 || sin_stride < 0) return XATTN_ERR_SHAPE;
  if (cos_stride % 8 || sin_stride % 8 || !a16(q) || !a16(k) || !a16(cos) || !a16(sin)) return XATTN_ERR_ALIGN;
  RopeParams p;
  p.q = static_cast<__bf16*>(q);
  p.k = static_cast<__bf16*>(k);
  p.cos = static_cast<const __bf16*>(cos);
  p.sin = static_cast<const __bf16*>(sin);
  p.cos_sn = cos_stride;
  p.sin_sn = sin_stride;
  p.heads = num_heads;
  p.kv_heads = num_kv_heads;
  p.total = (int64_t)tokens * (num_heads + num_kv_heads) * 8;
  const int64_t grid = (p.total + 255) / 256;
  if (p.total / 8 > 0x7fffffff) return XATTN_ERR_SHAPE;
  hipLaunchKernelGGL(rope_kernel, dim3((unsigned)grid), dim3(256), 0, static_cast<hipStream_t>(stream), p);
  return hipGetLastError() == hipSuccess ? XATTN_OK : XATTN_ERR_LAUNCH;
}
