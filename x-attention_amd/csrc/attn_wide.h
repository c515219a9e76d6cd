// Block-sparse attention of few units: a workgroup of eight wavefronts per (head, q-block), two per 32 query rows, each of which has
// half of every tile's keys.  (The rule: in_wide in block_sparse_attn.hip.)
//
// Bound: with no more units than CUs a workgroup of four wavefronts is alone on its CU, one wavefront to a SIMD, and a tile is
// a chain of Q.K^T, softmax and P.V, of two barriers and of copies half a tile ahead: about 2.2 us where its matrix instructions and its
// fragment reads take 1 each.  Here a SIMD's two wavefronts have half of that chain each, side by side, and tiles of their own
// LDS (two K, two V and the queries: all 160 KiB) are copied a whole tile ahead, with one barrier per tile.  The halves' results
// meet in LDS at the end.  Calls, us: 1000 tokens of 32 / 8 heads 28.6 -> 27.0, 700 24.7 -> 23.2, 600 of 28 / 4 23.2 -> 22.2, 1000 of 32 / 32 at
// stride 8 29.9 -> 28.0.
#pragma once
#include "attn_rows32.h"

namespace xattn {

constexpr int kWideLds = 5 * kTileBytes;      // K, V of two stages, the q-block

// Rows 16 w .. 16 w + 15 of a tile by wavefront w of eight; the caller counts the four copies (wait_vm0).
__device__ __forceinline__ void copy_eighth(const __bf16* base, int64_t sn, int len, int kb, const int (&voff)[4], uint32_t tile, int wave) {
  const int rows_left = len - kb * kBlk;
  const int rows = rows_left < kBlk ? rows_left : kBlk;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(base + (int64_t)kb * kBlk * sn), 0, (int)((int64_t)rows * sn * 2), 0x00020000);
#pragma unroll
  for (int i = 0; i < 4; ++i) slab_copy_1k(rsrc, (uint32_t)voff[i], tile + (uint32_t)(wave * 4 + i) * 1024);
}
__device__ __forceinline__ void eighth_offsets(int64_t sn, int lane, int wave, int (&voff)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * (wave * 4 + i) + (lane >> 4);
    voff[i] = (int)(row * sn * 2) + (((lane & 15) ^ swz(row)) << 4);
  }
}

__global__ __launch_bounds__(512, 2) void block_sparse_wide_kernel(AttnParams p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  touch_params();
  Unit u;
  if (!find_work<true, false>(p, (int)blockIdx.x, u)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, hh = lane >> 5;
  const int rows = wave & 3, kh = wave >> 2;       // 32 rows of the q-block, half of a tile's keys; a SIMD has both halves
  const int n_blocks = u.n_blocks;
  const __bf16* kbase = p.k + (int64_t)u.kvh * p.k_sh;
  const __bf16* vbase = p.v + (int64_t)u.kvh * p.v_sh;
  const int q_pos = u.qb * kBlk + rows * 32 + r + p.kv_off;   // position of this lane's query token on the key axis
  const int last_pos = u.qb * kBlk + rows * 32 + 31 + p.kv_off;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char_ptr)lds;

  FragAddr la;
  frag_addressing(lane, la);
  int voffK[4], voffV[4];
  eighth_offsets(p.k_sn, lane, wave, voffK);
  eighth_offsets(p.v_sn, lane, wave, voffV);
  // tile j is in K at 2 (j % 2) tiles, V behind it
  auto copy = [&](int j, int kb) __attribute__((always_inline)) {
    const uint32_t at = lds0 + (uint32_t)((j & 1) * 2 * kTileBytes);
    copy_eighth(kbase, p.k_sn, p.Lk, kb, voffK, at, wave);
    copy_eighth(vbase, p.v_sn, p.Lk, kb, voffV, at + kTileBytes, wave);
  };
  {
    int voffQ[4];
    eighth_offsets(p.q_sn, lane, wave, voffQ);
    copy_eighth(p.q + (int64_t)u.head * p.q_sh, p.q_sn, p.Lq, u.qb, voffQ, lds0 + 4 * kTileBytes, wave);
  }
  int kb = u.kb, kb_next = u.kb_next;
  if (n_blocks > 0) copy(0, kb);

  f32x16 oacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[i][v] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  bf16x8 qreg[8];

  for (int j = 0; j < n_blocks; ++j) {
    // the list's next entry comes with the tile
    int kb_then = u.list[j + 2 < n_blocks ? j + 2 : j];
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");      // tile j is there, the other stage has been read
    asm volatile("" : "+s"(kb_then));
    if (j == 0) {
      const char* Qs = lds + 4 * kTileBytes + rows * 8192;
#pragma unroll
      for (int s = 0; s < 8; ++s) qreg[s] = *reinterpret_cast<const bf16x8*>(Qs + la.kaddr[s]);
    }
    if (j + 1 < n_blocks) copy(j + 1, kb_next);
    const char* Ks = lds + (j & 1) * 2 * kTileBytes + kh * 16384;
    const int key0 = kb * kBlk + kh * 64;
    if (key0 < p.Lk && (!p.causal || key0 <= last_pos)) {              // (else no row sees a key of this half)
      f32x16 sacc[2];
      qk_tile<2>(Ks, la.kaddr, qreg, sacc);
      if (key0 + 64 > p.Lk || (p.causal && key0 + 63 > u.qb * kBlk + rows * 32 + p.kv_off)) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) mask_step(sacc[nt], key0 + nt * 32, hh, q_pos, p.Lk, p.causal);
      }
      bf16x8 pfrag[4];
      softmax_tile<2>(sacc, oacc, m_run, l_run, p.scale_log2, pfrag);
      pv_tile<4>(Ks + kTileBytes, la.vaddr, pfrag, oacc);
    }
    kb = kb_next;
    kb_next = clamp_block(kb_then, p.nkb);
  }

  // the halves meet: the second key half's wavefronts leave theirs in the tiles
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  char* const o1 = lds + rows * 16384 + lane * 16;
  float* const ml = reinterpret_cast<float*>(lds + 2 * kTileBytes) + rows * 128 + lane;
  if (kh == 1) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      f32x4 w;
#pragma unroll
      for (int t = 0; t < 4; ++t) w[t] = oacc[i >> 2][(i & 3) * 4 + t];
      *reinterpret_cast<f32x4*>(o1 + i * 1024) = w;
    }
    ml[0] = m_run;
    ml[64] = l_run;
  }
  __syncthreads();
  if (kh == 0) {
    const float m1 = ml[0], m = fmaxf(m_run, m1), safe = m == -INFINITY ? 0.f : m;
    const float w0 = fast_exp2(m_run - safe), w1 = fast_exp2(m1 - safe);      // 0 where a half saw no key of this row
    l_run = w0 * l_run + w1 * ml[64];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const f32x4 o = *reinterpret_cast<const f32x4*>(o1 + i * 1024);
#pragma unroll
      for (int t = 0; t < 4; ++t) oacc[i >> 2][(i & 3) * 4 + t] = w0 * oacc[i >> 2][(i & 3) * 4 + t] + w1 * o[t];
    }
    store_out(p, u.head, u.qb, rows, lane, r, hh, oacc, l_run, lds + rows * 16384);
  }
}

}  // namespace xattn
