// Shared device helpers for the gfx950 XAttention kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace xattn {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2;

constexpr int kWave = 64;
constexpr int kHeadDim = 128;
constexpr float kLog2e = 1.4426950408889634f;
// Cache policy of a buffer load or store, "not temporal" (the instruction's nt bit): for what is read once, or not read
// again soon.  256 CUs stream 256 MiB at 6.2 to 6.4 TB/s with it, at 5.1 to 5.5 without, whatever is in flight beyond
// 16 KiB per CU.
constexpr int kNotTemporal = 2;

// D[32x32] += A[32x16] * B[16x32], bf16 in, fp32 accumulate.
// Lane l (r = l % 32, h = l / 32) supplies A[r][8h..8h+7] and B[8h..8h+7][r];
// it receives D[8*(v/4) + 4h + v%4][r] in element v of the accumulator.
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
  bf16x2 p;
  p[0] = (__bf16)lo;
  p[1] = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, p);
}

// waits until every outstanding global/buffer load of this wavefront (including
// loads that write LDS directly) has completed; LDS and scalar counters untouched
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// value held by the lane 32 positions away (the other half-wave)
__device__ __forceinline__ float swap_half(float x) { return __shfl_xor(x, 32, 64); }

// x combined with the value of the lane 32 positions away, in every lane.  One
// v_permlane32_swap exchanges the upper half of its first operand with the lower
// half of its second: fed two copies of x it leaves (lower half, lower half) in
// the first and (upper half, upper half) in the second - both partners in every
// lane, without a trip through the LDS crossbar.  Written as inline assembly
// (the compiler's builtin hands back the first result twice); the s_nop pairs
// cover the wait states the instruction needs after a VALU write of its
// operands and before a VALU read of its results.
__device__ __forceinline__ void half_pair(float x, float& lo, float& hi) {
  lo = x;
  hi = x;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(lo), "+v"(hi));
}
// Two values combined across the half-waves at once: the lower half-wave ends up with a of the lane plus a of its
// partner, the upper half-wave with b plus b of its partner - one swap where two half_sum() calls need two.
__device__ __forceinline__ float half_sum_pair(float a, float b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return a + b;
}
__device__ __forceinline__ float half_sum(float x) {
  float lo, hi;
  half_pair(x, lo, hi);
  return lo + hi;
}
__device__ __forceinline__ float half_max(float x) {
  float lo, hi;
  half_pair(x, lo, hi);
  return fmaxf(lo, hi);
}

// Reductions over the wavefront through the data-parallel lane moves: within rows of 16 lanes by shifts of 1, 2, 4 and 8,
// then over the rows; lane 63 ends up with the result, which comes back as a uniform value.  (A butterfly of lane permutes
// takes a trip through the LDS crossbar per step, about 700 clk for a search step of the selection.)
template <int kCtrl, int kRows>
__device__ __forceinline__ uint32_t lane_move(uint32_t old, uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)x, kCtrl, kRows, 0xf, false);
}
template <typename F>
__device__ __forceinline__ uint32_t wave_fold(uint32_t x, F f) {   // f idempotent: max or min
  x = f(x, lane_move<0x111, 0xf>(x, x));
  x = f(x, lane_move<0x112, 0xf>(x, x));
  x = f(x, lane_move<0x114, 0xf>(x, x));
  x = f(x, lane_move<0x118, 0xf>(x, x));
  x = f(x, lane_move<0x142, 0xa>(x, x));
  x = f(x, lane_move<0x143, 0xc>(x, x));
  return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}
__device__ __forceinline__ uint32_t wave_max(uint32_t x) {
  return wave_fold(x, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}
__device__ __forceinline__ uint32_t wave_min(uint32_t x) {
  return wave_fold(x, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
}
// sum of the lanes up to and including the lane's own
__device__ __forceinline__ int wave_scan(int x) {
  auto add = [](int a, uint32_t b) { return a + (int)b; };
  x = add(x, lane_move<0x111, 0xf>(0u, (uint32_t)x));
  x = add(x, lane_move<0x112, 0xf>(0u, (uint32_t)x));
  x = add(x, lane_move<0x114, 0xf>(0u, (uint32_t)x));
  x = add(x, lane_move<0x118, 0xf>(0u, (uint32_t)x));
  x = add(x, lane_move<0x142, 0xa>(0u, (uint32_t)x));
  return add(x, lane_move<0x143, 0xc>(0u, (uint32_t)x));
}

// largest value and sum of floats, in every lane
__device__ __forceinline__ float wave_maxf(float x) {
  auto f = [](uint32_t a, uint32_t b) { return __builtin_bit_cast(uint32_t, fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b))); };
  return __builtin_bit_cast(float, wave_fold(__builtin_bit_cast(uint32_t, x), f));
}
__device__ __forceinline__ float wave_sumf(float x) {
  auto add = [](float a, uint32_t b) { return a + __builtin_bit_cast(float, b); };
  x = add(x, lane_move<0x111, 0xf>(0u, __builtin_bit_cast(uint32_t, x)));
  x = add(x, lane_move<0x112, 0xf>(0u, __builtin_bit_cast(uint32_t, x)));
  x = add(x, lane_move<0x114, 0xf>(0u, __builtin_bit_cast(uint32_t, x)));
  x = add(x, lane_move<0x118, 0xf>(0u, __builtin_bit_cast(uint32_t, x)));
  x = add(x, lane_move<0x142, 0xa>(0u, __builtin_bit_cast(uint32_t, x)));
  x = add(x, lane_move<0x143, 0xc>(0u, __builtin_bit_cast(uint32_t, x)));
  return __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_readlane((int)__builtin_bit_cast(uint32_t, x), 63));
}

typedef __attribute__((address_space(3))) char* lds_char_ptr;

// one KiB of a slab of rows of 128 bytes (8 of them), global -> LDS; the caller counts it in vmcnt
__device__ __forceinline__ void slab_copy_1k(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(dst), "v"(voff), "s"(rsrc) : "memory", "m0");
}

}  // namespace xattn
