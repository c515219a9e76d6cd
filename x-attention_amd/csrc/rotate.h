// Rotary embedding in the registers of the projection kernels.  Rounds where the bf16 tensor expression
// q * cos + rotate_half(q) * sin rounds: after each product and after the sum.
#pragma once
#include "xattn_common.h"

namespace xattn {

__device__ __forceinline__ float bf16_round(float x) { return (float)(__bf16)x; }

// contraction would skip the roundings in between
#pragma clang fp contract(off)
__device__ __forceinline__ void rotate_pair(float& x0, float& x1, float c0, float c1, float s0, float s1) {
  const float a0 = bf16_round(x0 * c0) + bf16_round(-x1 * s0);
  const float a1 = bf16_round(x1 * c1) + bf16_round(x0 * s1);
  x0 = bf16_round(a0);
  x1 = bf16_round(a1);
}
#pragma clang fp contract(fast)

// What a token's chunks f .. f + 7 and f + 64 .. f + 71 are turned by; cs and sn point at the token's values of feature f
struct Turn {
  bf16x8 c0, c1, s0, s1;
};
__device__ __forceinline__ Turn turn_of(const __bf16* cs, const __bf16* sn) {
  return {*reinterpret_cast<const bf16x8*>(cs), *reinterpret_cast<const bf16x8*>(cs + 64), *reinterpret_cast<const bf16x8*>(sn),
          *reinterpret_cast<const bf16x8*>(sn + 64)};
}
// 16-byte chunks f .. f + 7 (y0) and f + 64 .. f + 71 (y1) of a head, f < 64
__device__ __forceinline__ void rotate_chunks(bf16x8& y0, bf16x8& y1, const Turn& t) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float a = (float)y0[e], b = (float)y1[e];
    rotate_pair(a, b, (float)t.c0[e], (float)t.c1[e], (float)t.s0[e], (float)t.s1[e]);
    y0[e] = (__bf16)a;
    y1[e] = (__bf16)b;
  }
}

}  // namespace xattn
