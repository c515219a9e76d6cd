// The projections of an attention layer for turns of up to about a thousand tokens: y = x W^T with rows as long as the
// hidden state; q, k and v in one launch with the rotation of q and k in its epilogue, or the output projection.
//
// Bound: with at most a tile per CU, by how fast one CU fills its LDS (a CU has 32 KiB of loads in flight, whatever is asked of
// it: at most 76 GB/s from memory, 130 from the L2), so the tile is the largest that still gives most CUs one: 64 x 64 up to 256
// tiles, then 64 tokens x 128 features, 128 x 128, 192 x 128 and, for q, k and v, 256 x 128.  CUs left over may pull the weights
// into the L2 (proj_pull.h; weights from memory: q, k, v of 64 tokens, 4096 wide, 22.9 -> 19.9 us, of 192 30.8 -> 23.1, of 512
// 40.8 -> 33.6; the output of 320, 5120 wide, 38.8 -> 30.9).  Whole products stay below those rates: the tiles of those 512 tokens
// copy 2.1 MB each, 51 GB/s without pullers and 62 with them, of 33 us 2 for the first slab, 27 in the loop, 3 in the epilogue: a
// step of 128 x 128 takes 830 clk, 640 without its copies, 512 of them MFMAs, whether fragments are read in full or halves.  The larger tiles took the place of two 128 x 128 ones per CU (4096 wide, 700 tokens 66 -> 45 us, 1000 72 -> 57,
// 1280 73 -> 63).  Splitting a step's depth over two groups of wavefronts helps the smallest tile only (17.6 -> 13.3 us at 64
// tokens), where the chain of 64 steps is the time; on the larger ones, where it would save a third of the LDS reads, it is 1 to 8 %
// slower.
//
// Library products against this kernel, weights from memory, one box, in turn, in captured graphs, us.  q, k, v (of the library three
// launches, without the rotation, which is 4 to 5 more) by tokens:
//   width, heads      64          200         500         700         1000        1280        1500
//   1024   8 + 2*8    34 / 7.6    32 / 7.3    32 / 9.5    34 / 12.2   34 / 13.1   35 / 14.5   36 / 17.3
//   2048   32 + 2*8   34 / 12.1   35 / 15.2   41 / 21     47 / 26.7   49 / 33     55 / 37     library
//   3584   28 + 2*4   40 / 17.9   41 / 21.7   48 / 29     67 / 33     71 / 44     81 / 50     82 / 55
//   4096   32 + 2*8   45 / 20.6   47 / 26     61 / 35     73 / 47     83 / 57     98 / 66     library
//   5120   40 + 2*8   59 / 27.3   59 / 36     87 / 50     103 / 57    116 / 77    library
//   8192   64 + 2*8   62 / 51     97 / 64     133 / 95    167 / 118   library
// Output (features x depth), by the same tokens: 1024 x 1024 8.3 / 5.6, 8 / 5.6, 8.5 / 5.8, 8.7 / 5.8, 8.8 / 6, 9.4 / 7.2,
// 9.4 / 7.3; 3072 x 3072 16 / 14.2, 17.4 / 13.3, 20.8 / 18.6, 25.6 / 22.1, 29.6 / 24.8, 33 / 29.6, 40 / 33.5; 4096 x 4096 15.7 /
// 18.5, 22.3 / 17.4, 29.6 / 27, 33 / 31, 42 / 36.5, 49 / 46, 52 / 51; 5120 x 5120 22.7 / 24.7, 29.4 / 28, 48 / 37, 52 / 44, 64
// / 57; 8192 x 8192 35 / 47, 56 / 50, 80 / 73, 99 / 94.  Up to 64 tokens there is a single row of tiles, each a chain over the
// whole depth, which the library splits; so it does where the features are fewer than the depth.  Such a turn is bound by the
// host's calls, though, and the library's is the dearer one: the whole layer, 4096 wide, on 6000 tokens with the library's output
// product / this kernel's before weights were pulled ahead, 2 tokens 70 / 62, 16 68 / 64, 64 68 / 74.5, 100 68 / 68.
#include "lds_limit.h"
#include "proj_pull.h"
#include "rotate.h"
#include "xattn_hip.h"

namespace xattn {

struct ProjParams {
  const __bf16* x;           // [tokens][K]
  const __bf16* w[3];        // weights, rows of K contiguous elements
  const __bf16* bias[3];     // or null
  __bf16* y[3];              // [tokens][features of the product]
  int64_t w_sn[3];           // row stride, elements
  int n[3];                  // features, multiples of 128 (0: no such product)
  int M, K;                  // tokens, depth (a multiple of 64)
  const __bf16* cos;         // [tokens][128]; products 0 and 1 are rotated (kRope)
  const __bf16* sin;
  int64_t cos_sn, sin_sn;
};

template <int kN, int kThreads, int kAhead>
__device__ __forceinline__ void pull_weights(const ProjParams& p, uint32_t mt, uint32_t total, uint32_t per_xcd) {
  PullLane l;
  const uint32_t lane = ((blockIdx.x >> 3) - per_xcd) * kThreads + threadIdx.x, lanes = ((gridDim.x >> 3) - per_xcd) * kThreads;
  if (!pull_lane(blockIdx.x & 7, lane, lanes, per_xcd, total, mt, kN, p.n[0], p.n[1], kAhead, &l)) return;
  const char* const row = reinterpret_cast<const char*>(p.w[l.product] + (int64_t)l.row * p.w_sn[l.product]);
  const uint32_t steps = (uint32_t)p.K / 64;
  for (uint32_t t = l.step; t < steps; t += 8 * l.every) {
    uint32_t v[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const uint32_t*>(row + (int64_t)(t + u * l.every < steps ? t + u * l.every : t) * 128);
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) asm volatile("" ::"v"(v[u]));
  }
}

// Four wavefronts (2 x 2) take 64 * NB features x 64 * MB tokens; 64-deep slabs of both operands go straight to a ring of NS
// LDS stages, NS - 1 steps ahead of their use, one barrier per step.  KS = 2: four more multiply the second half of each
// slab, and the two sums of every element are added at the end.  kPull: workgroups beyond the tiles pull weights (a kernel of its
// own, since the code ahead of the tiles' loop moves it: 1 to 3 % of a narrow product's time).
template <int NB, int MB, int NS, int KS, bool kRope, bool kPull>
__global__ __launch_bounds__(256 * KS, 2) void proj_gemm_kernel(ProjParams p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int kN = 64 * NB, kM = 64 * MB;
  constexpr int kStage = (kN + kM) * 128;           // bytes of one 64-deep step
  constexpr int kSubs = 4 / KS;                     // 16-deep sub-steps of a wavefront
  constexpr int kLoads = 2 * (NB + MB) / KS;        // KiB a wavefront copies per step: first W's, then x's
  constexpr int kLoadsW = 2 * NB / KS, kLoadsX = 2 * MB / KS;
  constexpr int kChunks = 8 * NB, kPairs = kChunks / 2;       // of a token in a tile, and rotation partners
  constexpr int kTurns = (kM * kPairs + 256 * KS - 1) / (256 * KS), kTurnsAhead = kTurns < 4 ? kTurns : 4;
  constexpr int kPer = (kLoads + kSubs - 2) / (kSubs - 1);   // ... and in each of its sub-steps but the last
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave >> 2, wn = (wave >> 1) & 1, wm = wave & 1;
  const int r = lane & 31, hh = lane >> 5;

  // Ids are dealt round-robin to the 8 XCDs; an XCD gets one contiguous run of tiles, token tiles fastest, so that the
  // weights - most of the bytes - enter one XCD's L2 only
  const uint32_t mt = (uint32_t)(p.M + kM - 1) / kM;
  const uint32_t total = mt * (uint32_t)((p.n[0] + p.n[1] + p.n[2]) / kN), per_xcd = (total + 7) / 8;
  const uint32_t lin = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per_xcd) {
    if (kPull) pull_weights<kN, 256 * KS, NS - 1>(p, mt, total, per_xcd);
    return;
  }
  if (lin >= total) return;
  int f0 = (int)(lin / mt) * kN, t3 = 0;
  const int m0 = (int)(lin % mt) * kM;
  if (kRope) {
    if (f0 >= p.n[0]) { f0 -= p.n[0]; t3 = 1; }
    if (t3 == 1 && f0 >= p.n[1]) { f0 -= p.n[1]; t3 = 2; }
  }
  // With 64 features a tile holds features 32j .. 32j + 31 of a head and their rotation partners 64 further on: 16-byte
  // chunk c of a tile's row is chunk feature_chunk(c) of the product's
  const int head_c = f0 / 128 * 16, j4 = f0 % 128 / 64 * 4;
  auto feature_chunk = [&](int c) __attribute__((always_inline)) { return head_c + (NB == 2 ? c : (c & 3) + j4 + (c >> 2) * 8); };

  const int64_t w_snb = p.w_sn[t3] * 2;
  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc((void*)(p.w[t3] + (int64_t)head_c * 8 * p.w_sn[t3]), 0, (int)(128 * w_snb), 0x00020000);
  const int rows_left = p.M - m0;
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.x + (int64_t)m0 * p.K), 0, (rows_left < kM ? rows_left : kM) * p.K * 2, 0x00020000);
  // a lane's part of a copied KiB: row lane / 8 of 8, chunk lane % 8 of the slab, stored at c ^ ((row >> 1) & 7)
  const int rl = lane >> 3, c = lane & 7;
  uint32_t voff[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const bool is_w = i < kLoadsW;
    const int row = is_w ? (wave * kLoadsW + i) * 8 + rl : (wave * kLoadsX + i - kLoadsW) * 8 + rl;
    const int src = is_w ? (feature_chunk(row >> 3) - head_c) * 8 + (row & 7) : row;
    voff[i] = (uint32_t)src * (uint32_t)(is_w ? w_snb : (int64_t)p.K * 2) + (uint32_t)((c ^ ((row >> 1) & 7)) << 4);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char_ptr)lds;
  const int steps = p.K / 64;
  // Tiles that share weights or tokens ask for a slab at the same time, and all of them wait for the memory's answer.  Nobody pulling
  // for them, each takes every four slabs in another order, so that it waits for one of them and finds three in the L2 (weights from
  // memory, us: output of 500 tokens, 4096 wide, 29.0 / 25.5, of 1000 38.4 / 36.1; q, k, v of 320 31.2 / 26.7; 5120 wide, output of
  // 700 44.9 / 43.2; 8192 wide, q, k, v of 130 55.9 / 53.6).  Orders of eight slabs give the same, of two a third of it; a quarter of the depth apart for each token tile, slabs leave the L2
  // between two uses (35 / 42).  Not with pulled weights (-7 to +7 %), 64 x 64 tiles (2 % slower), nor 256 tokens (2 to 5 % slower).
  constexpr bool kShift = !kPull && NB == 2 && MB <= 2 && NS == 4;
  const int shift = kShift ? (int)(lin % mt + lin / mt) & 3 : 0, whole = steps & ~3;
  auto slab_of = [&](int t) __attribute__((always_inline)) { return kShift && t < whole ? (t & ~3) | ((t + shift) & 3) : t; };
  // (the steps of a ring's first fill may be more than there are: such a copy moves nothing, its offset being outside the resource;
  // the last steps issue none, since it would cost the CU 20 clk all the same)
  auto copy_piece = [&](int t, int st, int i, bool is_step) __attribute__((always_inline)) {
    const bool is_w = i < kLoadsW;
    const uint32_t dst = lds0 + (uint32_t)st * kStage + (is_w ? (uint32_t)(wave * kLoadsW + i) : (uint32_t)(kN / 8 + wave * kLoadsX + i - kLoadsW)) * 1024;
    slab_copy_1k(is_w ? wres : xres, is_step ? voff[i] + (uint32_t)slab_of(t) * 128 : 0xffffffffu, dst);
  };
  f32x16 acc[NB][MB];
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;
  const int sw = (r >> 1) & 7;
  bf16x8 fa[2][NB], fb[2][MB];
  auto read = [&](int st, int s, int buf) __attribute__((always_inline)) {
    const char* at = lds + st * kStage + r * 128 + (((2 * (s + wk * kSubs) + hh) ^ sw) << 4);
#pragma unroll
    for (int a = 0; a < NB; ++a) fa[buf][a] = *reinterpret_cast<const bf16x8*>(at + (wn * NB + a) * 4096);
#pragma unroll
    for (int b = 0; b < MB; ++b) fb[buf][b] = *reinterpret_cast<const bf16x8*>(at + kN * 128 + (wm * MB + b) * 4096);
  };
#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) copy_piece(t, t, i, t < steps);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 2) * kLoads) : "memory");
  read(0, 0, 0);
  // A step is four sub-steps of NB * MB MFMAs; the fragments of the next sub-step and the copies of step t + NS - 1 are
  // issued between them.  The barrier sits before the last sub-step's MFMAs: by then this wavefront has read every
  // fragment of step t and its copies of step t + 1 have landed, so behind it step t + 1 may be read and step t's stage
  // refilled.
  // `left`: the steps behind step t + 1 whose copies have been issued; kLanded: every copy has landed.  The counts are of
  // copies alone, which are written here in assembly: a load that the compiler issues or moves can only make a wait stricter.
  constexpr int kLanded = -1;
  int st = 0, t = 0;
  auto step = [&](auto copies, auto left) __attribute__((always_inline)) {
    const int next = st + 1 == NS ? 0 : st + 1, fill = st == 0 ? NS - 1 : st - 1;
#pragma unroll
    for (int s = 0; s < kSubs; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      if (s == kSubs - 1) {
        if constexpr (decltype(left)::value == kLanded) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(decltype(left)::value * kLoads) : "memory");
        read(next, 0, 0);     // (a repeat of old data behind the last step)
      } else {
        read(st, s + 1, (s + 1) & 1);
#pragma unroll
        for (int i = s * kPer; decltype(copies)::value && i < kLoads && i < (s + 1) * kPer; ++i) copy_piece(t + NS - 1, fill, i, true);
      }
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[a][b] = mfma32(fa[s & 1][a], fb[s & 1][b], acc[a][b]);
    }
    st = next;
    ++t;
  };
  while (t < steps - (NS - 1)) step(std::true_type(), std::integral_constant<int, NS - 2>());
  const int ch = tid % kPairs, feature = feature_chunk(ch) * 8;      // its partner is 64 further on
  auto token = [&](int i) __attribute__((always_inline)) { return (i * 256 * KS + tid) / kPairs; };
  auto turn_at = [&](int i) __attribute__((always_inline)) {
    const int64_t m = m0 + (token(i) < rows_left ? token(i) : 0);
    return turn_of(p.cos + m * p.cos_sn + feature % 128, p.sin + m * p.sin_sn + feature % 128);
  };
  auto last = [&](auto left) __attribute__((always_inline)) {
    if (t < steps) step(std::false_type(), left);
  };
  static_assert(NS >= 2 && NS <= 6, "the steps behind the last copy are written for these");
  if constexpr (NS >= 6) last(std::integral_constant<int, 3>());
  if constexpr (NS >= 5) last(std::integral_constant<int, 2>());
  if constexpr (NS >= 4) last(std::integral_constant<int, 1>());
  if constexpr (NS >= 3) last(std::integral_constant<int, 0>());
  // With a step left or none every copy has landed, unless there were fewer steps than the first fill has stages: then those that move
  // nothing may be under way still.
  if (steps < NS - 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // The cosines and sines of the first four tokens that this lane turns are on their way while the last step multiplies.  (Asked
  // for one token after the other behind the exchange, a layer's 500 tokens took 35.0 us instead of 34.0, 1000 63.8 instead of 61.3; ahead of
  // the last three steps, whose waits then have to count them, 34.5 as here and 58.2 instead of 58.0.)
  Turn turns[kTurnsAhead];
  if (kRope) {
#pragma unroll
    for (int i = 0; i < kTurnsAhead; ++i) turns[i] = turn_at(i);
    __builtin_amdgcn_sched_barrier(0);
  }
  last(std::integral_constant<int, kLanded>());
  // every copy has landed and every fragment has been read: the LDS takes the tile, token-major, chunk c of token m at
  // c ^ (m & (chunks - 1))
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  static_assert((KS - 1) * 4 * NB * MB * 4096 + kM * kN * 2 <= NS * kStage, "the halves' sums and the tile");
  char* const tile = lds + (KS - 1) * 4 * NB * MB * 4096;
  if (KS == 2) {
    f32x4* const half = reinterpret_cast<f32x4*>(lds + (wave & 3) * NB * MB * 4096) + lane;
#pragma unroll
    for (int i = 0; i < NB * MB * 4; ++i) {
      f32x16& x = acc[i / 4 / MB][i / 4 % MB];
      if (wk == 1) half[i * 64] = f32x4{x[i % 4 * 4], x[i % 4 * 4 + 1], x[i % 4 * 4 + 2], x[i % 4 * 4 + 3]};
    }
    __syncthreads();
    if (wk == 0) {
#pragma unroll
      for (int i = 0; i < NB * MB * 4; ++i) {
        f32x16& x = acc[i / 4 / MB][i / 4 % MB];
        const f32x4 o = half[i * 64];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[i % 4 * 4 + u] += o[u];
      }
    }
  }
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (wk) continue;
      const int ch = (wn * NB + a) * 4 + g;          // features 8 ch + 4 hh .. + 3 of the tile
      float bs[4] = {0.f, 0.f, 0.f, 0.f};
      if (p.bias[t3]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) bs[u] = (float)p.bias[t3][feature_chunk(ch) * 8 + hh * 4 + u];
      }
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        const int m = (wm * MB + b) * 32 + r;
        u32x2 o;
        o[0] = pack_bf16(acc[a][b][g * 4 + 0] + bs[0], acc[a][b][g * 4 + 1] + bs[1]);
        o[1] = pack_bf16(acc[a][b][g * 4 + 2] + bs[2], acc[a][b][g * 4 + 3] + bs[3]);
        *reinterpret_cast<u32x2*>(tile + m * (kN * 2) + ((ch ^ (m & (kChunks - 1))) << 4) + hh * 8) = o;
      }
    }
  __syncthreads();
  // kPairs lanes write a token's
  __bf16* const y = p.y[t3];
  const int64_t y_sn = p.n[t3];
#pragma unroll
  for (int i = 0; i < kTurns; ++i) {
    const int m = token(i);
    if (m >= kM || m >= rows_left) break;
    const char* row = tile + m * (kN * 2);
    bf16x8 y0 = *reinterpret_cast<const bf16x8*>(row + ((ch ^ (m & (kChunks - 1))) << 4));
    bf16x8 y1 = *reinterpret_cast<const bf16x8*>(row + (((ch + kPairs) ^ (m & (kChunks - 1))) << 4));
    if (kRope && t3 < 2) {
      rotate_chunks(y0, y1, turns[i % kTurnsAhead]);
      if (i + kTurnsAhead < kTurns) turns[i % kTurnsAhead] = turn_at(i + kTurnsAhead);
    }
    __bf16* const at = y + (int64_t)(m0 + m) * y_sn + feature;
    *reinterpret_cast<bf16x8*>(at) = y0;
    *reinterpret_cast<bf16x8*>(at + 64) = y1;
  }
}

}  // namespace xattn

using namespace xattn;

namespace {
bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// The tile for `features` features of `tokens` tokens (see the head of the file), or none: the products are large enough
// for the library.  An output product of 256-token tiles would only tie with it (1500 to 2000 tokens, 4096 wide: 54 to 63 us,
// library 51 to 60), q, k and v are three of its launches.  Token counts that miss 256 tiles by the rounding (2600 tokens of
// 3072 features: 504 tiles of 128 x 128, 264 of 128 x 256) have two workgroups per CU.
enum Tile { kNone, k64x64, k128x64, k128x128, k128x192, k128x256, k128x128Twice };
constexpr unsigned kCUs = 256;
Tile tile_for(int64_t tokens, int64_t features, bool qkv) {
  auto tiles = [&](int n, int m) { return features / n * ((tokens + m - 1) / m); };
  if (tiles(64, 64) <= kCUs) return k64x64;
  if (tiles(128, 64) <= kCUs) return k128x64;
  if (tiles(128, 128) <= kCUs) return k128x128;
  if (tiles(128, 192) <= kCUs) return k128x192;
  if (!qkv) return kNone;
  if (tiles(128, 256) <= kCUs) return k128x256;
  return tiles(128, 128) <= 2 * kCUs ? k128x128Twice : kNone;
}

template <int NB, int MB, int NS, int KS, bool kRope, bool kPull>
int launch_tiles(const ProjParams& p, unsigned grid, hipStream_t s) {
  constexpr int kLds = (NB + MB) * 64 * 128 * NS;
  static_assert(kLds <= 160 * 1024, "LDS of a CU");
  static LdsLimit limit;
  if (limit.raise((const void*)proj_gemm_kernel<NB, MB, NS, KS, kRope, kPull>) != hipSuccess) return XATTN_ERR_LAUNCH;
  hipLaunchKernelGGL((proj_gemm_kernel<NB, MB, NS, KS, kRope, kPull>), dim3(grid), dim3(256 * KS), kLds, s, p);
  return hipGetLastError() == hipSuccess ? XATTN_OK : XATTN_ERR_LAUNCH;
}

// kMayPull: one workgroup per CU, and the rule of proj_pull.h gains
template <int NB, int MB, int NS, int KS, bool kRope, bool kMayPull>
int launch(const ProjParams& p, hipStream_t s) {
  const unsigned tiles = (unsigned)((p.M + 64 * MB - 1) / (64 * MB)) * (unsigned)((p.n[0] + p.n[1] + p.n[2]) / (64 * NB));
  const unsigned grid = (tiles + 7) / 8 * 8, places = pull_places((uint32_t)p.M, 64 * MB, 64 * NB, tiles);
  if (kMayPull && places) return launch_tiles<NB, MB, NS, KS, kRope, kMayPull>(p, grid + 8 * places, s);
  return launch_tiles<NB, MB, NS, KS, kRope, false>(p, grid, s);
}

// offsets inside a tile are held in 32 bits
bool shape_ok(int tokens, int width) { return tokens > 0 && width >= 64 && width % 64 == 0 && width <= 65536; }
bool stride_ok(int64_t sn, int width) { return sn >= width && sn <= ((int64_t)1 << 22); }

template <bool kRope>
int run(const ProjParams& p, void* stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  const Tile tile = tile_for(p.M, (int64_t)p.n[0] + p.n[1] + p.n[2], kRope);
  if (tile == k64x64) return launch<1, 1, 6, 2, kRope, true>(p, s);
  if (tile == k128x64) return launch<2, 1, 4, 1, kRope, true>(p, s);
  if (tile == k128x128) return launch<2, 2, 4, 1, kRope, true>(p, s);
  if (tile == k128x192) return launch<2, 3, 4, 1, kRope, true>(p, s);
  if constexpr (kRope) {        // (tile_for: q, k and v alone)
    if (tile == k128x256) return launch<2, 4, 3, 1, kRope, true>(p, s);
    if (tile == k128x128Twice) return launch<2, 2, 2, 1, kRope, false>(p, s);
  }
  return XATTN_ERR_SHAPE;
}
}  // namespace

extern "C" int xattn_proj_gemm_fits(int tokens, int width, int features, int qkv) {
  return shape_ok(tokens, width) && features >= 128 && features % 128 == 0 && tile_for(tokens, features, qkv != 0) != kNone;
}

extern "C" int xattn_qkv_rope_gemm(const void* x, int tokens, int width, const void* wq, int64_t wq_stride, const void* bq,
                                   const void* wk, int64_t wk_stride, const void* bk, const void* wv, int64_t wv_stride,
                                   const void* bv, const void* cos, const void* sin, int64_t cos_stride, int64_t sin_stride,
                                   void* q, void* k, void* v, int num_heads, int num_kv_heads, int head_dim, void* stream) {
  if (!x || !wq || !wk || !wv || !cos || !sin || !q || !k || !v) return XATTN_ERR_NULL;
  if (head_dim != kHeadDim) return XATTN_ERR_HEAD_DIM;
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads > 4096 || num_kv_heads > 4096) return XATTN_ERR_HEADS;
  if (!shape_ok(tokens, width) || !stride_ok(wq_stride, width) || !stride_ok(wk_stride, width) || !stride_ok(wv_stride, width) ||
      cos_stride < 0 || sin_stride < 0)
    return XATTN_ERR_SHAPE;
  if (wq_stride % 8 || wk_stride % 8 || wv_stride % 8 || cos_stride % 8 || sin_stride % 8) return XATTN_ERR_ALIGN;
  for (const void* a : {x, wq, wk, wv, cos, sin, (const void*)q, (const void*)k, (const void*)v})
    if (!a16(a)) return XATTN_ERR_ALIGN;
  ProjParams p{};
  p.x = static_cast<const __bf16*>(x);
  const void *w[3] = {wq, wk, wv}, *b[3] = {bq, bk, bv};
  void* y[3] = {q, k, v};
  const int64_t sn[3] = {wq_stride, wk_stride, wv_stride};
  const int n[3] = {num_heads, num_kv_heads, num_kv_heads};
  for (int i = 0; i < 3; ++i) {
    p.w[i] = static_cast<const __bf16*>(w[i]);
    p.bias[i] = static_cast<const __bf16*>(b[i]);
    p.y[i] = static_cast<__bf16*>(y[i]);
    p.w_sn[i] = sn[i];
    p.n[i] = n[i] * kHeadDim;
  }
  p.M = tokens;
  p.K = width;
  p.cos = static_cast<const __bf16*>(cos);
  p.sin = static_cast<const __bf16*>(sin);
  p.cos_sn = cos_stride;
  p.sin_sn = sin_stride;
  return run<true>(p, stream);
}

extern "C" int xattn_gemm(const void* x, int tokens, int width, const void* w, int64_t w_stride, const void* bias, void* y,
                          int features, void* stream) {
  if (!x || !w || !y) return XATTN_ERR_NULL;
  if (!shape_ok(tokens, width) || !stride_ok(w_stride, width) || features < 128 || features % 128) return XATTN_ERR_SHAPE;
  if (w_stride % 8 || !a16(x) || !a16(w) || !a16(y)) return XATTN_ERR_ALIGN;
  ProjParams p{};
  p.x = static_cast<const __bf16*>(x);
  p.w[0] = static_cast<const __bf16*>(w);
  p.bias[0] = static_cast<const __bf16*>(bias);
  p.y[0] = static_cast<__bf16*>(y);
  p.w_sn[0] = w_stride;
  p.n[0] = features;
  p.M = tokens;
  p.K = width;
  return run<false>(p, stream);
}
