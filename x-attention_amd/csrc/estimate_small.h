// The estimator's MFMA pass for launches that leave the 256x256 tiles of estimate_gemm_kernel mostly empty: short
// prompts, and chunks of a few hundred tokens on top of a long cache.  Same scores, same partial results, to the bit.
//
// A workgroup of four wavefronts takes 128 keys (one softmax tile) x 32 * MT query rows; wavefront w computes the scores
// of keys 32w .. 32w+31 against all rows.  Where a head has fewer rows than that, the rows of several heads of the KV
// group share a tile (`pack`), so that every key is read once per group.  64-deep slabs of both operands go straight to
// a ring of NS LDS stages (buffer loads that write LDS), NS - 1 steps ahead of their use (NS with MT 1), one barrier per step.
//
// Bound: with at most a tile per CU the time is the chain of 2 * stride steps - 0.16 us each with MT 1, the barrier, the
// dependent MFMAs and the fragment reads of a step, against 1.4 us of a 256x256 step.  With more tiles per CU two workgroups share it
// and the copies into LDS (about 50 bytes per clock and CU) and the fragment reads (1 + MT per MT MFMAs) are the limit:
// 0.55 (MT 2) and 0.65 (MT 4) of the flop rate of the large tiles.
#pragma once
#include "estimate_params.h"
#include "select_row.h"

namespace xattn {

// kSelect (MT 1, rows that see no key past the first softmax tile): normalisation and selection follow in the same
// workgroup, which has whole rows.  A 1000-token prompt then takes one launch of 11.8 us instead of two of 9.2 and 7.0.
template <int RBS, int MT, int NS, bool kSelect>
__global__ __launch_bounds__(256, 2) void estimate_small_kernel(EstParams p, SelParams sp) {
  static_assert(!kSelect || MT == 1, "the selection takes a wavefront per query block of 32 rows");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int kKeys = kSub, kRows = 32 * MT;
  constexpr int kStage = (kKeys + kRows) * 128;     // bytes of one 64-deep step
  constexpr int kLoads = 4 + MT;                    // KiB a wavefront copies per step
  constexpr int kPer = (kLoads + 2) / 3;            // ... and in each of the step's first three sub-steps
  constexpr bool kAhead = MT == 1;
  static_assert(kAhead ? NS == 4 : NS <= 3, "the steps behind the last copy are written for these");
  constexpr int kPer4 = (kLoads + 3) / 4;           // ... or (kAhead) in each of four
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, hh = lane >> 5;

  // Tile of this workgroup.  Ids are dealt round-robin to the 8 XCDs; an XCD gets one contiguous run of tiles, ordered by
  // KV group, query-tile row, key tile, head set, so that it works on few KV heads and the sets share a key tile.
  const uint32_t G = (uint32_t)(p.H / p.Hkv), sets = (G + p.pack - 1) / (uint32_t)p.pack;
  const uint32_t per_group = (uint32_t)p.tiles_per_head * sets, total = per_group * (uint32_t)p.Hkv;
  const uint32_t per_xcd = (total + 7) / 8;
  const uint32_t lin = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  for (int i = (int)blockIdx.x * 256 + tid; i < p.clear_words; i += (int)gridDim.x * 256) p.clear[i] = 0;
  if (lin >= total) return;
  const uint32_t g = lin / per_group, rem = lin - g * per_group;
  const uint32_t set = rem % sets;
  int tt = (int)(rem / sets), m0 = p.row_begin, n0 = 0, hi_tile = 0;
  for (;; m0 += p.tile_rows) {
    const int mlast = m0 + p.tile_rows - 1 < p.live_end ? m0 + p.tile_rows - 1 : p.live_end - 1;
    hi_tile = row_hi(p, mlast);
    int last = hi_tile / kSub;
    last = last < p.nNT - 1 ? last : p.nNT - 1;
    const int first = row_lo(p, m0) / kSub;
    const int cnt = last - first + 1;
    if (tt < cnt || m0 + p.tile_rows >= p.live_end) {
      n0 = (first + tt) * kSub;
      break;
    }
    tt -= cnt;
  }
  const int h0 = (int)(g * G + set * (uint32_t)p.pack);
  const int h_end = (int)((g + 1) * G);

  // operands: K' slab rows 32w..32w+31 are copied by the wavefront that multiplies them, and not at all when none of
  // its keys is visible; tokens past the real length read as zeros
  const int64_t k_snb = p.k_sn * 2, q_snb = p.q_sn * 2;
  const int n_w = n0 + wave * 32;                   // first key of this wavefront
  const bool live_w = n_w <= hi_tile && n_w < p.n_rk;
  const int64_t tok0 = (int64_t)n0 * p.S, left = p.Lk - tok0, span = (int64_t)kKeys * p.S;
  const int64_t krows = left < 0 || !live_w ? 0 : (left < span ? left : span);
  const __amdgpu_buffer_rsrc_t kres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.k + (int64_t)g * p.k_sh + (krows > 0 ? tok0 * p.k_sn : 0)), 0, (int)(krows * k_snb), 0x00020000);
  const __amdgpu_buffer_rsrc_t qres = __builtin_amdgcn_make_buffer_rsrc((void*)(p.q + (int64_t)h0 * p.q_sh + (int64_t)m0 * p.S * p.q_sn), 0, 0x7fffffff, 0x00020000);
  // slab row of a lane: instruction i of K' covers rows 32w + 8i + lane / 8, of Q' rows 8 (w MT + i) + lane / 8; 16-byte
  // chunk c of row r sits at c ^ ((r >> 1) & 7) (conflict-free fragment reads)
  const int rl = lane >> 3, c = lane & 7;
  uint32_t voffK[4], voffQ[MT];
  int qtok[MT];                                     // token of the row at reshape offset 0; past the end: never valid
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = wave * 32 + i * 8 + rl;
    voffK[i] = (uint32_t)((int64_t)row * p.S * k_snb) + (uint32_t)((c ^ ((row >> 1) & 7)) << 4);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int row = (wave * MT + i) * 8 + rl;
    const int hs = row >> p.tile_shift, m = m0 + (row & (p.tile_rows - 1));
    const bool ok = m < p.live_end && h0 + hs < h_end;
    qtok[i] = ok ? m * p.S : 0x40000000;
    voffQ[i] = (uint32_t)((int64_t)hs * p.q_sh * 2 + (int64_t)(m - m0) * p.S * q_snb) + (uint32_t)((c ^ ((row >> 1) & 7)) << 4);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char_ptr)lds;
  const int steps = p.S * 2;
  // Piece j of step t: 0 .. 3 are K' (not copied by a wavefront whose keys nobody sees), then Q'.  The last steps copy nothing
  // and wait for fewer: a copy of 1 KiB costs the CU about 20 clk also where its offset is outside the resource.
  auto copy_piece = [&](int t, int j) __attribute__((always_inline)) {
    const int i = t >> 1;
    const uint32_t st = lds0 + (uint32_t)(t % NS) * kStage;
    if (j < 4) {
      const uint32_t ko = (uint32_t)(i * (int)k_snb + (t & 1) * 128);
      slab_copy_1k(kres, voffK[j] + ko, st + (uint32_t)(wave * 4 + j) * 1024);
    } else {
      const int qi = p.S - 1 - i;
      const uint32_t qo = (uint32_t)(qi * (int)q_snb + (t & 1) * 128);
      slab_copy_1k(qres, qtok[j - 4] + qi < p.Lq ? voffQ[j - 4] + qo : 0xffffffffu,
                   st + 16384 + (uint32_t)(wave * MT + j - 4) * 1024);
    }
  };
  f32x16 acc[MT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[a][v] = 0.f;
  const int swz = (r >> 1) & 7;
  if (kAhead) {
    // A step's fragments are read together, a step ahead of its MFMAs: a sub-step is one MFMA of 32 clk, an answer of the LDS
    // takes four times that, and with fragments read a sub-step ahead every sub-step waited for it (1000 tokens, stride 16, estimate
    // and selection 13.2 -> 11.8 us; with MT 2, two MFMAs and more workgroups to a CU, no difference).  The barrier of step t: this
    // wavefront has step t's fragments in registers and its copies of step t + 1 have landed, so behind it step t + 1 may be read and
    // step t's stage refilled.
    const int from = live_w ? 0 : 4;
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int j = 0; j < kLoads; ++j)
        if (j >= from) copy_piece(t, j);
    if (live_w) {
      bf16x8 fa[2][4], fb[2][4][MT];
      auto read = [&](int t, int buf) __attribute__((always_inline)) {
        const char* st = lds + (t % NS) * kStage;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int ch = ((2 * s + hh) ^ swz) << 4;
          fa[buf][s] = *reinterpret_cast<const bf16x8*>(st + (wave * 32 + r) * 128 + ch);
#pragma unroll
          for (int a = 0; a < MT; ++a) fb[buf][s][a] = *reinterpret_cast<const bf16x8*>(st + 16384 + (a * 32 + r) * 128 + ch);
        }
      };
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * kLoads) : "memory");
      read(0, 0);
      // `left`: the steps behind step t + 1 that have been copied
      auto step = [&](int t, int buf, auto copies, auto left) __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(decltype(left)::value * kLoads) : "memory");
        read(t + 1, buf ^ 1);        // (a repeat of old data behind the last step)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
          for (int a = 0; a < MT; ++a) acc[a] = mfma32(fa[buf][s], fb[buf][s][a], acc[a]);
#pragma unroll
          for (int j = s * kPer4; decltype(copies)::value && j < kLoads && j < (s + 1) * kPer4; ++j) copy_piece(t + NS, j);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      int t = 0;
      for (; t < steps - NS; t += 2) {      // (steps = 2 S)
        step(t, 0, std::integral_constant<int, 1>(), std::integral_constant<int, 2>());
        step(t + 1, 1, std::integral_constant<int, 1>(), std::integral_constant<int, 2>());
      }
      step(t, 0, std::integral_constant<int, 0>(), std::integral_constant<int, 2>());
      step(t + 1, 1, std::integral_constant<int, 0>(), std::integral_constant<int, 1>());
      step(t + 2, 0, std::integral_constant<int, 0>(), std::integral_constant<int, 0>());
      step(t + 3, 1, std::integral_constant<int, 0>(), std::integral_constant<int, 0>());
    } else {
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * MT) : "memory");
      int t = 0;
      for (; t < steps - NS; ++t) {
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 2) * MT) : "memory");
#pragma unroll
        for (int j = 4; j < kLoads; ++j) copy_piece(t + NS, j);
      }
      for (; t < steps; ++t) asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    }
  } else
  // A step is four sub-steps of MT MFMAs; the fragments of the next sub-step and the copies of step t + NS - 1 are issued
  // between them.  The barrier sits before the last sub-step's MFMAs: by then this wavefront has read every fragment of
  // step t and its copies of step t + 1 have landed, so behind it step t + 1 may be read and step t's stage refilled.
  if (live_w) {
#pragma unroll
    for (int t = 0; t < NS - 1; ++t)
#pragma unroll
      for (int j = 0; j < kLoads; ++j) copy_piece(t, j);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 2) * kLoads) : "memory");
    bf16x8 fa[2], fb[2][MT];
    auto read = [&](int t, int s, int buf) __attribute__((always_inline)) {
      const char* st = lds + (t % NS) * kStage;
      const int ch = ((2 * s + hh) ^ swz) << 4;
      fa[buf] = *reinterpret_cast<const bf16x8*>(st + (wave * 32 + r) * 128 + ch);
#pragma unroll
      for (int a = 0; a < MT; ++a) fb[buf][a] = *reinterpret_cast<const bf16x8*>(st + 16384 + (a * 32 + r) * 128 + ch);
    };
    read(0, 0, 0);
    auto step = [&](int t, auto copies) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        __builtin_amdgcn_sched_barrier(0);
        if (s == 3) {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(decltype(copies)::value ? (NS - 2) * kLoads : 0) : "memory");
          read(t + 1, 0, 0);     // (a repeat of old data behind the last step)
        } else {
          read(t, s + 1, (s + 1) & 1);
#pragma unroll
          for (int j = s * kPer; decltype(copies)::value && j < kLoads && j < (s + 1) * kPer; ++j) copy_piece(t + NS - 1, j);
        }
#pragma unroll
        for (int a = 0; a < MT; ++a) acc[a] = mfma32(fa[s & 1], fb[s & 1][a], acc[a]);
      }
    };
    int t = 0;
    for (; t < steps - NS + 1; ++t) step(t, std::integral_constant<int, 1>());
    for (; t < steps; ++t) step(t, std::integral_constant<int, 0>());
  } else {
#pragma unroll
    for (int t = 0; t < NS - 1; ++t)
#pragma unroll
      for (int j = 4; j < kLoads; ++j) copy_piece(t, j);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 2) * MT) : "memory");
    int t = 0;
    for (; t < steps - NS + 1; ++t) {
#pragma unroll
      for (int j = 4; j < kLoads; ++j) copy_piece(t + NS - 1, j);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 2) * MT) : "memory");
    }
    for (; t < steps; ++t) asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  }
  // every copy has landed and every fragment has been read: the LDS is free for the exchange below
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // ---- epilogue, in the operations and the order of estimate_gemm_kernel: there one wavefront has all 128 keys of a
  // row; here the four wavefronts' maxima and sums meet in LDS
  float* maxes = reinterpret_cast<float*>(lds);                 // [4][kRows]
  float* parts = maxes + 4 * kRows;                             // [4][2][MT][64]
  float* psum = parts + 8 * MT * 64;                            // kSelect: [128 / RBS][32] partial block sums,
  float* row_m = psum + (kSub / RBS) * 32;                      // row maxima
  float* row_inv = row_m + 32;                                  // and 1 / row sums
  float mx[MT];
#pragma unroll
  for (int a = 0; a < MT; ++a) {
    const int m = m0 + ((a * 32 + r) & (p.tile_rows - 1));
    const int lo = row_lo(p, m), hi = row_hi(p, m);
    const int at = n_w + hh * 4, last = (hi < p.n_rk - 1 ? hi : p.n_rk - 1) - at;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[a][v] = (v >> 2) * 8 + (v & 3) <= last ? acc[a][v] : -INFINITY;
    if (p.own_chunk_only) {
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][v] = (v >> 2) * 8 + (v & 3) >= lo - at ? acc[a][v] : -INFINITY;
    }
    float w = -INFINITY;
#pragma unroll
    for (int v = 0; v < 16; ++v) w = fmaxf(w, acc[a][v]);
    w = half_max(w * p.scale_log2);
    if (hh == 0) maxes[wave * kRows + a * 32 + r] = w;
  }
  __syncthreads();
  const int kb_first = n0 / RBS, kb_left = p.nkb - kb_first;
#pragma unroll
  for (int a = 0; a < MT; ++a) {
    const int rr = a * 32 + r;
    mx[a] = fmaxf(fmaxf(maxes[rr], maxes[kRows + rr]), fmaxf(maxes[2 * kRows + rr], maxes[3 * kRows + rr]));
    const float safe = mx[a] == -INFINITY ? 0.f : mx[a];
    const int head = h0 + (rr >> p.tile_shift), m = m0 + (rr & (p.tile_rows - 1));
    const bool row_ok = m < p.live_end && head < h_end;
    float* const prow = p.P + partial_at(p, row_ok ? head : h0, row_ok ? m - p.row_begin : 0) + (int64_t)kb_first * kStrip;
    const bool st0 = row_ok && hh == 0, st1 = row_ok && hh == 1;
    auto put = [&](int k, bool on, float x) __attribute__((always_inline)) {
      if (kSelect) {
        if (on) psum[k * 32 + r] = x;
      } else if (k < kb_left && on) {
        prow[k * kStrip] = x;
      }
    };
    float s[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      s[q] = 0.f;
#pragma unroll
      for (int u = 0; u < 4; ++u) s[q] += fast_exp2(__builtin_fmaf(acc[a][q * 4 + u], p.scale_log2, -safe));
    }
    float* const part = parts + (wave * 2 * MT + a) * 64 + lane;
    constexpr int Gk = RBS / 8;
    if (Gk == 1) {
#pragma unroll
      for (int q2 = 0; q2 < 2; ++q2) {
        const float both = half_sum_pair(s[2 * q2], s[2 * q2 + 1]);
        part[q2 * MT * 64] = both;
        const int k = wave * 4 + 2 * q2;
        put(k, st0, both);
        put(k + 1, st1, both);
      }
    } else if (Gk == 2) {
      const float both = half_sum_pair(s[0] + s[1], s[2] + s[3]);
      part[0] = both;
      const int k = wave * 2;
      put(k, st0, both);
      put(k + 1, st1, both);
    } else {
      const float all = half_sum(s[0] + s[1] + s[2] + s[3]);
      part[0] = hh == 0 ? all : 0.f;
      put(wave, st0, all);
    }
  }
  __syncthreads();
#pragma unroll
  for (int a = 0; a < MT; ++a) {
    if (a % 4 != wave) continue;
    const int rr = a * 32 + r;
    const int head = h0 + (rr >> p.tile_shift), m = m0 + (rr & (p.tile_rows - 1));
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int q2 = 0; q2 < (RBS == 8 ? 2 : 1); ++q2) tot += parts[((w * 2 + q2) * MT + a) * 64 + lane];
    tot = half_sum(tot);
    if (kSelect) {
      const float Mw[4] = {mx[a], -INFINITY, -INFINITY, -INFINITY}, Lw[4] = {tot, 0.f, 0.f, 0.f};
      if (hh == 0) stat_combine(Mw, Lw, m < p.live_end && head < h_end && m < p.real_rows, 0, &row_m[r], &row_inv[r]);
    } else if (m < p.live_end && head < h_end && hh == 0) {
      const int64_t at = ((int64_t)head * p.nT + n0 / kSub) * p.rows + (m - p.row_begin);
      p.Mt[at] = mx[a];
      p.Lt[at] = tot;
    }
  }
  if (kSelect) {
    __syncthreads();
    // wavefront b: query block b of the tile
    const int head = h0 + ((wave * RBS) >> p.tile_shift), m = m0 + ((wave * RBS) & (p.tile_rows - 1));
    if (wave * RBS >= 32 || head >= h_end || m >= p.live_end) return;
    const size_t wave_bytes = (size_t)sp.npow2 * 8 + ((sp.nkb + 15) & ~15);
    char* mine = reinterpret_cast<char*>(row_inv + 32) + wave * wave_bytes;
    float* xs = reinterpret_cast<float*>(mine + (size_t)sp.npow2 * 8 - (size_t)((sp.nkb + 15) & ~15) * 4);
    // lane (kb, l): rows 4l .. 4l+3 of the block, summed as estimate_select_kernel does
    constexpr int kLanes = RBS / 4;
    const int l = lane % kLanes, kb = lane / kLanes;
    const int m4 = m + l * 4, row4 = wave * RBS + l * 4;
    int hi = row_hi(p, m4);
    hi = hi < p.n_rk - 1 ? hi : p.n_rk - 1;
    float sum = 0.f;
    if (kb < kSub / RBS && kb <= hi / RBS) {
      const f32x4 rM = *reinterpret_cast<const f32x4*>(row_m + row4);
      sum = group_sum4(*reinterpret_cast<const f32x4*>(psum + kb * 32 + row4), rM, rM, *reinterpret_cast<const f32x4*>(row_inv + row4));
    }
    sum = sum_lanes<kLanes>(sum, lane);
    if (l == 0 && kb < kSub / RBS && kb < sp.nkb) xs[kb] = sum;
    for (int c = kSub / RBS + lane; c < sp.nkb; c += 64) xs[c] = 0.f;
    __builtin_amdgcn_wave_barrier();
    const int row = m / RBS;
    if (sp.sums_out) store_sums(sp, xs, head, row, lane);
    select_row<kSub / RBS>(sp, xs, head, row, reinterpret_cast<uint64_t*>(mine), reinterpret_cast<uint8_t*>(mine + (size_t)sp.npow2 * 8), lane);
  }
}

}  // namespace xattn
