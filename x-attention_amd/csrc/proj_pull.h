// What CUs without a tile of a projection do: they pull the weights of their XCD's tiles into its L2, ahead of the tiles
// (proj_gemm.hip).  The rule and the lanes' shares, for the host too.
//
// A CU has at most 32 KiB of loads in flight and gets them back in order, so a tile's fill runs at 32 KiB per latency of the
// slowest load among them: 76 GB/s where each step's weights come from memory, 130 where they are in the L2.  (Loads by the
// tile's own CU don't help: they queue with the others.  Nor does the scalar cache, some 27 ns per line.)
#pragma once
#include "xattn_common.h"

namespace xattn {

constexpr uint32_t kCUsPerXcd = 32;

// CUs of an XCD that pull for `tiles` tiles of tile_tokens x tile_features, or none.  An XCD has per_xcd tiles, which read the
// weights of per_xcd / mt tiles' features.  Times are us, weights from memory, without / with:
//  - A CU pulls 76 GB/s, about what a tile of a single row of tiles takes in, and half of what several share.  Where the idle CUs
//    are fewer than that takes, they end long after the tiles: 2 tokens, 12288 wide, 224 tiles 74 / 242; 2, 8192 wide, 160 tiles
//    39.7 / 47; 128, 5120 wide, 224 tiles 31 / 37; 192 (output), 240 tiles 28 / 45.
//  - Beyond that, more of them help where the weights are most of a tile (128 features x 64 tokens: twice as many, 0.80 of the
//    time without any instead of 0.86 over 23 sizes), and elsewhere only stand in the way of the tiles' own loads.  For a single
//    row of tiles three quarters: 64 tokens, 4096 wide, with 20, 12 and 9 CUs of each XCD 21.4, 20.9, 20.9 (22.5 without), and if the weights
//    are in the memory-side cache, as of a small model, 18.2, 17.1, 15.7 (14.5 without); the output with 24, 8 and 6 19.6, 19.0,
//    19.1 (21.3) and 16.0, 14.0, 13.5 (13.5).
//  - A last token tile that lacks rows asks for less, runs ahead and has pulled some of the weights for the others already, which
//    leaves less to gain: output of 3072 features, 330 tokens 20.8 / 16.9, 1000 31.6 / 25.5, of 5120 200 33.5 / 26.9; q, k, v of 4096
//    wide, 72 tokens 18.2 / 17.8, 400 33.4 / 32.5 (of whole tiles 128 22.7 / 20.2, 512 40.8 / 34).
__host__ __device__ inline uint32_t pull_places(uint32_t tokens, uint32_t tile_tokens, uint32_t tile_features, uint32_t tiles) {
  const uint32_t mt = (tokens + tile_tokens - 1) / tile_tokens, per_xcd = (tiles + 7) / 8;
  if (per_xcd >= kCUsPerXcd) return 0;
  const uint32_t idle = kCUsPerXcd - per_xcd;
  if (mt == 1 ? idle <= per_xcd : 2 * idle * mt < per_xcd) return 0;
  const uint32_t shared = (per_xcd + mt - 1) / mt;
  const uint32_t wanted = mt == 1 ? (3 * per_xcd + 3) / 4 : tile_features > tile_tokens ? 2 * shared : shared;
  return idle < wanted ? idle : wanted;
}

struct PullLane {
  int product, row;       // of which weight matrix, and which of its rows
  uint32_t step, every;   // 64-deep steps step, step + every, ...
};
// Lane `lane` of the `lanes` that pull for XCD xcd takes one row of its tiles' (heads of 128 features, whole), and every `every`-th
// step from `ahead` on; false: none.
__host__ __device__ inline bool pull_lane(uint32_t xcd, uint32_t lane, uint32_t lanes, uint32_t per_xcd, uint32_t total, uint32_t mt,
                                          uint32_t tile_features, int n0, int n1, uint32_t ahead, PullLane* l) {
  const uint32_t first = xcd * per_xcd;
  if (first >= total) return false;
  const uint32_t last = (first + per_xcd < total ? first + per_xcd : total) - 1;
  const uint32_t head0 = first / mt * tile_features / 128, heads = last / mt * tile_features / 128 + 1 - head0;
  const uint32_t rows = heads * 128;
  l->every = lanes / rows;
  if (lane >= l->every * rows) return false;
  l->row = (int)(head0 * 128 + lane % rows);
  l->product = 0;
  if (l->row >= n0) { l->row -= n0; l->product = 1; }
  if (l->product == 1 && l->row >= n1) { l->row -= n1; l->product = 2; }
  l->step = ahead + lane / rows;
  return true;
}

}  // namespace xattn
