// What the estimator's kernels share: the launch parameters and the visibility rule of a reshaped query row.
#pragma once
#include "xattn_common.h"

namespace xattn {

constexpr int kSub = 128;        // keys of a softmax tile: what one (maximum, sum) pair covers

struct EstParams {
  const __bf16* q;
  const __bf16* k;
  int64_t q_sh, q_sn, k_sh, k_sn;
  float* P;        // [H][nkb][rows]  partial block sums relative to the tile maximum
  float* Mt;       // [H][nT][rows]   tile maximum (exp2 domain)
  float* Lt;       // [H][nT][rows]   tile sum
  float* scores;   // optional [H][n_rq][n_rk] raw scores
  float* sums;     // output block sums: [H][win_rows][nkb], q-block row i stored at row i - win_row0
  int win_row0, win_rows;
  int H, Hkv, Lq, Lk, S, rbs;
  int n_rq, n_rk, nkb, nqb, nT;
  int rcs;                  // reshaped keys per chunk
  int kdb;                  // query-row subsampling: query row m stands for reshaped row m * kdb
  int rcs_q, rbs_q;         // query rows per chunk / per query block (rcs / kdb, rbs / kdb)
  int row_begin, row_end;   // query rows handled by this call
  int live_end;             // rows at or past it give zero block sums (padding) or are not asked for: never computed
  int rows;                 // live_end - row_begin (pitch of P / Mt / Lt)
  int nT_real;              // 128-key tiles from here on hold padded keys only (nT when causal): not computed either
  int off;                  // position of reshaped row 0 on the key axis: n_rk - n_rq * kdb
  int real_rows;            // query rows >= real_rows give all-zero block sums
  int causal, own_chunk_only;
  int no_softmax;           // block sums of exp(scaled score) instead of softmax probabilities
  float scale_log2;
  // Depth slabs of the reshaped GEMM.  Slab j multiplies query token
  // m*S + (pairs[j] >> 4) with key token n*S + (pairs[j] & 15); n_pairs = 0 means
  // the S pairs (S-1-i, i) of the antidiagonal reshape, in closed form.
  int n_pairs;
  uint8_t pairs[64];
  int nMT, nNT;             // tile rows over [row_begin, row_end) / tile columns over n_rk
  int tiles_per_head;       // tiles with a visible pair, per head
  int64_t total_tiles;      // tiles_per_head * H
  // estimate_small_kernel: a tile's rows are tile_rows rows of each of pack heads of one KV group
  unsigned long long* clear;   // clear_words words set to zero for the passes that follow
  int pack, tile_rows, tile_shift;   // powers of two, tile_rows = 1 << tile_shift
  // estimate_gemm_kernel with packed rows: quarters of 64 rows per head, 256-row tiles per KV group, first key tile, key tiles
  int quarters, group_tiles, first_key_tile, key_tiles;
  // estimate_gemm_kernel with half tiles: tiles taken whole, tiles behind them taken as two halves of 128 rows, and per head
  // the tiles (of keys from first_key_tile on) of a last row tile that has one half
  int whole_tiles, split_tiles, last_row_tiles;
  int clear_words;
};

// Place of row `rel` (counted from row_begin) in P, for key block 0; the next key block's is kStrip on.  Strips of 32 rows, key
// block after key block: what a workgroup of the selection reads lies together, and a wavefront of the estimate writes two key
// blocks of its rows with one store at a constant offset.  Key block after key block with all rows of each, the selection read
// 128 bytes every 4 * rows and half a wavefront wrote at a time (us, that way / this way: estimate and selection of 131072
// tokens 3831 / 3790, of 15000 153.5 / 149; selection alone of 32768 52 / 48, of a video of 65536 160 / 147).
constexpr int kStrip = 32;
__host__ __device__ inline int strips_of(int rows) { return (rows + kStrip - 1) / kStrip; }
__device__ __forceinline__ int64_t partial_at(const EstParams& p, int head, int rel) {
  return (int64_t)(head * strips_of(p.rows) + rel / kStrip) * p.nkb * kStrip + rel % kStrip;
}

// first / last visible reshaped key of reshaped query row m
// (with kdb > 1 the row's causal limit is that of the LAST reshaped row of its
// group, xattn/src/Xattention.py:217-222, while its tokens are those of the first, :88-93)
__host__ __device__ inline int row_lo(const EstParams& p, int m) {
  return (p.causal && p.own_chunk_only) ? (m / p.rcs_q) * p.rcs + p.off : 0;
}
__host__ __device__ inline int row_hi(const EstParams& p, int m) {
  return p.causal ? m * p.kdb + p.kdb - 1 + p.off : p.n_rk - 1;
}

// The arithmetic of the normalisation, shared by the stand-alone pass and the fused forms so that all give the same bits (fixed operation order, no contraction into fused multiply-adds).
#pragma clang fp contract(off)
// folds tile T's maximum / sum into a running (M, L)
__device__ __forceinline__ void stat_step(float& M, float& L, float mt, float lt) {
  const float Mn = fmaxf(M, mt);
  const float safe = (Mn == -INFINITY) ? 0.f : Mn;
  L = L * fast_exp2(M - safe) + lt * fast_exp2(mt - safe);
  M = Mn;
}
// combines the four partial (M, L) of a row (tiles T = first + w, + 4, ... for w = 0..3) into the row's
// maximum (0 when the row sees nothing, or without softmax) and 1 / sum (0 for rows that give zeros)
__device__ __forceinline__ void stat_combine(const float (&Mw)[4], const float (&Lw)[4], bool real_row, int no_softmax,
                                             float* rowM, float* rowInv) {
  const float Mr = fmaxf(fmaxf(Mw[0], Mw[1]), fmaxf(Mw[2], Mw[3]));
  const float safe = (Mr == -INFINITY) ? 0.f : Mr;
  float Lr = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) Lr += Lw[w] * fast_exp2(Mw[w] - safe);
  const bool real = real_row && Lr > 0.f;
  // without softmax the partial sums are referred to 2^0 and left unnormalised
  *rowM = no_softmax ? 0.f : safe;
  *rowInv = real ? (no_softmax ? 1.f : 1.f / Lr) : 0.f;
}
// normalised partial sums of four consecutive rows, added up: the weights of the tile, and the sums of a key block with them
__device__ __forceinline__ f32x4 tile_weights(const f32x4& mt, const f32x4& rM, const f32x4& rI) {
  f32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = fast_exp2(mt[i] - rM[i]) * rI[i];
  return w;
}
__device__ __forceinline__ float weighted_sum4(const f32x4& pv, const f32x4& w, const f32x4& rI) {
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) acc += (rI[i] != 0.f) ? pv[i] * w[i] : 0.f;
  return acc;
}
__device__ __forceinline__ float group_sum4(const f32x4& pv, const f32x4& mt, const f32x4& rM, const f32x4& rI) {
  return weighted_sum4(pv, tile_weights(mt, rM, rI), rI);
}
#pragma clang fp contract(fast)

}  // namespace xattn
