// Projections and rotary embedding of an attention layer: what surrounds the prefill and decode kernels in the
// reference's Llama forward (xattn/src/load_llama.py:119-150, 207-218).
//
//  gemv_kernel: y = W x for ONE token, q, k and v in one launch with their rotation, or the output projection.  Bound by HBM:
//    every weight is read once and used once, 84 MB for a 4096-wide layer with 32 + 2 * 8 heads.  Four weight rows (for q
//    and k two rotary pairs d, d + 64 and their neighbours, so that the rotation happens in registers) are a workgroup's, a
//    quarter of their length each wavefront's, which requests all of it at once (up to 8192 elements) and is done: all loads
//    of a launch are asked for as soon as there is a place, the CUs get equal shares, and the chip is busy to the end.  With
//    four whole rows per wavefront, two batches of loads in flight, 4096 wide layers had 384 and 256 workgroups for 256
//    CUs.  us, weights from memory, q, k and v / output, then / now: 1024 wide 5.1 / 4.2 and 3.8 / 2.9, 2048 8.6 / 5.7 and 6.6 / 5.2,
//    4096 12.2 / 8.7 and 9.9 / 7.4 (5.1 TB/s), 5120 18.4 / 15.9 and 13.9 / 10.3, 8192 37.3 / 31.8 and 27.6 / 23.1; weights in the
//    memory-side cache, both, 4096 19.5 and 18.3, 5120 31.4 and 25.4.  (Two wavefronts per unit 0.6 slower, eight 2; what the last
//    thread needs requested ahead of the weights or behind them 0.5 to 1 slower.)  proj_gemm.hip has the products of more tokens.
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

constexpr int kGemvWaves = 4;

// A workgroup has one unit of four rows and its wavefronts every fourth chunk of 512 elements each, kBatch of them at once.
// kRope: a unit is rows d, d+1, d+64, d+65 of one head (products 0 and 1 rotated, 2 not); otherwise four rows in order
template <bool kRope, int kBatch, bool kNt>
__global__ __launch_bounds__(64 * kGemvWaves) void gemv_kernel(GemvParams p) {
  __shared__ __attribute__((aligned(16))) float sums[kGemvWaves][4];      // (written 16 bytes at a time)
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int unit = blockIdx.x, t = 0;
  if (kRope) {
    if (unit >= p.units[0]) { unit -= p.units[0]; t = 1; }
    if (t == 1 && unit >= p.units[1]) { unit -= p.units[1]; t = 2; }
  }
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

  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  const int chunks = (p.K + 511) / 512;
  for (int c0 = wave; c0 < chunks; c0 += kGemvWaves * kBatch) {
    u32x4 wv[kBatch][4], xv[kBatch];
#pragma unroll
    for (int c = 0; c < kBatch; ++c) {
      const int off = ((c0 + c * kGemvWaves) * 64 + lane) * 16;
      xv[c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xres, off, 0, 0));
#pragma unroll
      for (int i = 0; i < 4; ++i)
        wv[c][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wres[i], off, 0, kNt ? kNotTemporal : 0));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kBatch; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[i] = __builtin_fmaf(bf16_lo(wv[c][i][e]), bf16_lo(xv[c][e]), acc[i]);
          acc[i] = __builtin_fmaf(bf16_hi(wv[c][i][e]), bf16_hi(xv[c][e]), acc[i]);
        }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = wave_sumf(acc[i]);
  if (lane == 0) *reinterpret_cast<f32x4*>(sums[wave]) = f32x4{acc[0], acc[1], acc[2], acc[3]};
  __syncthreads();
  if (threadIdx.x == 0) {
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      y[i] = bf16_round(sums[0][i] + sums[1][i] + sums[2][i] + sums[3][i] + (p.bias[t] ? (float)p.bias[t][row[i]] : 0.f));
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
  rotate_chunks(y0, y1, turn_of(cs, sn));
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

// Bytes of a launch's weights from which they are loaded not temporal: from memory they come 5 to 8 % faster so (us, q, k and v /
// output, 4096 wide 10.7 / 8.0 -> 9.9 / 7.4, 8192 30.5 / 24.8 -> 27.6 / 23.1), and a model of such layers does not fit the memory-side cache
// (a single one that is run again and again does: 5120 wide 24.7 -> 25.4, 4096 equal, 8192 56 -> 50).  Narrower ones may (1024 wide, output,
// 2.9 -> 3.1).
constexpr int64_t kGemvNtBytes = 24 << 20;
constexpr int kMostUnits = 1 << 22;      // of a launch: a grid has fewer than 2^32 threads

template <bool kRope>
int launch_gemv(const GemvParams& p, int units, void* stream) {
  const int each = (p.K + 512 * kGemvWaves - 1) / (512 * kGemvWaves);      // chunks of a wavefront
  const bool nt = (int64_t)units * 4 * p.K * 2 > kGemvNtBytes;
  auto kernel = each == 1 ? gemv_kernel<kRope, 1, false> : each == 2 ? gemv_kernel<kRope, 2, false> : gemv_kernel<kRope, 4, false>;
  if (nt) kernel = each == 1 ? gemv_kernel<kRope, 1, true> : each == 2 ? gemv_kernel<kRope, 2, true> : gemv_kernel<kRope, 4, true>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)units), dim3(64 * kGemvWaves), 0, static_cast<hipStream_t>(stream), p);
  return hipGetLastError() == hipSuccess ? XATTN_OK : XATTN_ERR_LAUNCH;
}
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
  return launch_gemv<true>(p, units, stream);
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
  p.K = width;
  for (int done = 0; done < rows; done += 4 * kMostUnits) {
    const int units = (rows - done) / 4 < kMostUnits ? (rows - done) / 4 : kMostUnits;
    p.units[0] = units;
    if (const int rc = launch_gemv<false>(p, units, stream)) return rc;
    if (rows - done <= 4 * kMostUnits) break;      // (done may not pass the largest int)
    p.w[0] += 4 * (int64_t)kMostUnits * w_stride;
    p.y[0] += 4 * kMostUnits;
    if (p.bias[0]) p.bias[0] += 4 * kMostUnits;
  }
  return XATTN_OK;
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
