// Block-sparse attention with 64 query rows per wavefront, for long lists (all_rows64 and lists_decide have the rule).
//
// One workgroup of two wavefronts per (head, q-block), two workgroups per CU: each wavefront has a SIMD to itself, 424 to 465
// of its 512 registers, and nothing but its own instruction order to keep the matrix pipe busy while it exponentiates.  So a sweep
// is a software pipeline of steps of 32 keys: beside the scores of the next step and the output of the last one - 16 MFMAs
// each, alternating - the 32 exponentials of this step's scores are dealt out between the MFMAs, with the fragment reads of
// five pairs of MFMAs ahead and the copies of the tiles (global -> LDS) of the next 64 keys.
//
// Bound: MFMA, under the power limit.  Why 64 rows: a K or V fragment read from LDS serves twice the MFMAs that it serves in
// the 32-row kernel, whose LDS and vector pipes are shared by two wavefronts per SIMD.  Dense causal attention of 32768
// tokens, 32/8 heads, both on one box: 7.5 ms -> 6.65 ms (1.17 -> 1.32 PFLOP/s; MFMA busy 63 -> 75 % of SIMD cycles at 1.72 ->
// 1.6 GHz).  A wave tile of 64 x 128 takes 5150 clk for 4096 of MFMA; without fragment reads and copies 4590, without what
// keeps the order of instructions (pin, settle, MFMAs as assembly) 6200 - the compiler bunches the exponentials.
// A unit costs 3.9 us per CU beside its tiles, against 3.1 with 32 rows, where the other workgroup's wavefronts use the SIMD
// while this one waits for its first tiles: lists of 1, 2, 3, 8, 32 blocks 6.0, 7.0, 8.4, 16.3, 53 us per unit and CU,
// against 4.8, 6.4, 8.0, 17.0, 58 - a workgroup per unit.  With a queue (attn_unit.h) workgroups stay and go from unit to unit,
// whose queries and first keys are requested before the results of the last one leave; 0.8 us lie between two units.  Whole
// calls, ms, without / with: 131072 tokens 13.45 / 12.85, video of 65536 16.84 / 15.88, a field of 119056 141.7 / 137.8.
#pragma once
#include <type_traits>

#include "attn_unit.h"

namespace xattn {

// LDS of a workgroup: two halves of 64 keys of K, two of V, each 16 KiB, a half by its parity in the sweep.
constexpr int kHalfBytes = 64 * 256;
constexpr int kVAt = 2 * kHalfBytes;
constexpr int kLdsBytes = 4 * kHalfBytes;

// A lane's byte offset in load i of 4 rows of a tile whose rows are row_bytes apart, without the rows ahead of the load.
__device__ __forceinline__ uint32_t load_lane(uint32_t row_bytes, int lane, int i) {
  return (uint32_t)(lane >> 4) * row_bytes + (uint32_t)(((lane & 15) ^ swz(4 * i + (lane >> 4))) << 4);
}
// Loads 0 .. 7 are this wavefront's rows of the first half, 8 .. 15 those of the second; odd ones carry 1024 in the
// instruction (copy_2k).
__device__ __forceinline__ void tile_loads(uint32_t row_bytes, int lane, int wave, uint32_t (&voff)[16]) {
#pragma unroll
  for (int i = 0; i < 16; ++i)
    voff[i] = load_lane(row_bytes, lane, i & 3) + ((uint32_t)wave * 32 + (uint32_t)((i >> 3) * 64 + 4 * (i & 7))) * row_bytes - (uint32_t)(i & 1) * 1024;
}

struct LaneAddr : FragAddr {
  uint32_t voffK[16], voffV[16]; // copy of a tile, load by load
};

// Buffer resource of key block kb of one head (rows past the sequence end read as zeros), block_bytes = 128 rows.
__device__ __forceinline__ u32x4 block_resource(const __bf16* base, uint32_t block_bytes, uint32_t last_bytes, int kb, int nkb) {
  const uint64_t at = (uint64_t)base + (uint64_t)(uint32_t)kb * block_bytes;
  u32x4 r;
  r[0] = (uint32_t)at;
  r[1] = (uint32_t)(at >> 32);                 // (stride 0: addresses have 48 bits)
  r[2] = kb + 1 < nkb ? block_bytes : last_bytes;
  r[3] = 0x00020000;
  return r;
}

constexpr int kAhead = 5;
// Rows' reference maxima are moved once a lane's sum of the 32 probabilities of a step, 16 of each of two rows, is beyond
// kOutgrown.  So a probability is at most 2^8, as in the 32-row kernel, and where scores grow the largest of a row is brought
// back to 1, which bf16 holds exactly.  (Maxima 2^24 above the scores, moved beyond 2^24, are hardly ever moved and save up to
// 2 % - field of 8000 tokens 757 / 745 us, 60000 35210 / 35370, video of 65536 15530 / 15480 - but the error of the field's output
// against 64 bits is then 2.10e-3, with 32 rows 2.05e-3, this way 2.03e-3; values from 2^104 on overflow, below 2^-100 they lose
// bits.)
constexpr float kOutgrown = 0x1p8f;
constexpr float kNoKey = -3.402823466e+38f;   // reference maximum of a row that has seen no key

// What a sweep keeps in registers: 64 query rows of a wavefront as two groups of 32.
struct SweepState {
  f32x16 s[2][2];      // scores of a step of 32 keys: [step parity][row group]
  u32x4 p[2][2][2];    // its probabilities, packed bf16: [step parity][row group][16 keys]
  f32x16 o[2][4];      // output accumulators
  float m[2], l[2];    // reference maximum (times scale_log2) and this lane's share of the row sum
  bf16x8 kf[8];        // fragments of pairs of MFMAs, requested kAhead pairs ahead
  i16x4 vf[8][2];
};

// The MFMAs of a sweep, issued from assembly: scores in vector registers, outputs and queries in accumulator registers (the
// compiler keeps all of one kind and moves the others to and fro).  It knows no wait states for them: what reads a result
// outside the MFMAs stands behind settle().
__device__ __forceinline__ void mfma_first(f32x16& s, const bf16x8& k, const bf16x8& q) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(k), "a"(q));
}
__device__ __forceinline__ void mfma_score(f32x16& s, const bf16x8& k, const bf16x8& q) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(k), "a"(q));
}
__device__ __forceinline__ void mfma_out(f32x16& o, const bf16x8& v, const u32x4& p) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(o) : "v"(v), "v"(p));
}
__device__ __forceinline__ void settle() { asm volatile("s_nop 15\n\ts_nop 3" ::: "memory"); }
// ... and is named, or its first use might be moved ahead
__device__ __forceinline__ void settle(f32x16& a, f32x16& b) { asm volatile("s_nop 15\n\ts_nop 3" : "+v"(a), "+v"(b)); }
__device__ __forceinline__ void settle(f32x16 (&o)[2][4]) {
  asm volatile("s_nop 15\n\ts_nop 3" : "+a"(o[0][0]), "+a"(o[0][1]), "+a"(o[0][2]), "+a"(o[0][3]), "+a"(o[1][0]), "+a"(o[1][1]), "+a"(o[1][2]), "+a"(o[1][3]));
}

__device__ __forceinline__ bf16x8 join(const i16x4& a, const i16x4& b) {
  typedef __attribute__((__vector_size__(8 * sizeof(short)))) short i16x8;
  i16x8 x;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    x[u] = a[u];
    x[4 + u] = b[u];
  }
  return __builtin_bit_cast(bf16x8, x);
}

// Online softmax in the exp2 domain of the scores of a step, row group g, with the reference maxima of all its rows brought up
// to date (of none but those that have outgrown theirs, the others are soon the cause of another such step: us that way /
// this way, field 4000 271 / 257, 8000 775 / 757, video 18000 1320 / 1294, 65536 15720 / 15530).
__device__ __forceinline__ void softmax_slow(SweepState& w, int set, int g, float scale_log2, float& psum) {
  float mx = -INFINITY;
#pragma unroll
  for (int v = 0; v < 16; ++v) mx = fmaxf(mx, w.s[set][g][v]);
  mx = half_max(mx) * scale_log2;
  const float m_new = fmaxf(w.m[g], mx);
  const float alpha = fast_exp2(w.m[g] - m_new);
  w.m[g] = m_new;
  w.l[g] *= alpha;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) {
    asm volatile("" : "+a"(w.o[g][dt]));     // (sixteen vector registers at a time: those of the fast path stay where they are)
#pragma unroll
    for (int v = 0; v < 16; ++v) w.o[g][dt][v] *= alpha;
    asm volatile("" : "+a"(w.o[g][dt]));
  }
  psum = 0.f;
#pragma unroll
  for (int v = 0; v < 16; v += 2) {
    const float e0 = fast_exp2(__builtin_fmaf(w.s[set][g][v], scale_log2, -m_new));
    const float e1 = fast_exp2(__builtin_fmaf(w.s[set][g][v + 1], scale_log2, -m_new));
    psum = psum + e0 + e1;
    w.p[set][g][v >> 3][(v & 7) >> 1] = pack_bf16(e0, e1);
  }
}

// One load of part of a tile (1 KiB: 4 rows), global -> LDS, issued from assembly (the compiler would make the transposing
// reads wait for every such load it knows of); the caller waits with vmcnt.
__device__ __forceinline__ void copy_1k(const u32x4& rs, uint32_t voff, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(dst), "v"(voff), "s"(rs) : "memory", "m0");
}
// Two of them in a row, to base + kAt: the offset of 1024 counts on both sides, so the second one's voff is 1024 less.
template <int kAt>
__device__ __forceinline__ void copy_2k(const u32x4& rs, uint32_t voff0, uint32_t voff1, uint32_t base) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %3, 0 offen lds\n\t"
               "buffer_load_dwordx4 %2, %3, 0 offen offset:1024 lds" ::"s"(base), "v"(voff0), "v"(voff1), "s"(rs), "n"(kAt) : "m0", "scc");
}
__device__ __forceinline__ void pack_to(uint32_t& p, float lo, float hi) { asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(p) : "v"(lo), "v"(hi)); }
// Keeps an instruction where it stands in the text (the compiler would move it to its first use, or up to its operands).
__device__ __forceinline__ void pin(float& x) {
  asm volatile("" : "+v"(x));
  __builtin_amdgcn_sched_barrier(0);
}

// Buffer resources of the blocks being copied.
struct Copies {
  u32x4 k, v;
  uint32_t lds;                // this wavefront's share of the first half of K
};

// How far the softmax of a step's 32 scores per lane has come behind its m-th MFMA: exponentials taken.  They are done four
// MFMAs before the end, so that what the sums decide is known while the last ones run.
constexpr int exps_by(int m) { return m <= 0 ? 0 : m >= 26 ? 32 : m * 32 / 26; }
constexpr int args_by(int m) { return exps_by(m) + 2 < 32 ? exps_by(m) + 2 : 32; }
constexpr int packs_by(int m) { return exps_by(m - 1) / 2; }       // pairs packed
constexpr int sums_by(int m) { return exps_by(m - 2); }            // probabilities summed up

// A step of the sweep: scores of the next 32 keys (kQK), softmax of this step's (set kSet), output of the last step's
// probabilities (kPV), sixteen MFMAs of each kind side by side with the 32 exponentials.
// kK, kV: LDS offsets of the keys of the QK and PV of this step; kKn, kVn: of the next step's (-1: none).
// kBar: the next step starts on other halves of K and V: a barrier publishes them before their first fragment is requested.
// kFree: a second barrier, behind the last fragment of the present halves, lets the next step copy over them.
// kHk, kHv: halves of K and V that this step copies (-1: none).
template <int kSet, int kK, int kV, int kKn, int kVn, bool kQK, bool kPV, bool kBar, bool kFree, int kHk, int kHv>
__device__ __forceinline__ void sweep_step(SweepState& w, const bf16x8 (&q)[2][8], const char* lds, const LaneAddr& la, float scale_log2, const Copies& cp) {
  float t[32], e[32], psum[2];
  // The softmax behind MFMA m.  What is not vector arithmetic - fragment reads, copies - comes straight after the MFMA, the sum
  // ahead of the exponential: a read that follows vector instructions costs a wavefront alone on its SIMD 6 clk more (probe
  // of this loop without copies, clk per pair of 4 MFMAs: 135 this way, 139 to 143 in other orders of the arithmetic, 156 with
  // the reads behind it).
  auto softmax = [&](auto mc) __attribute__((always_inline)) {
    constexpr int m = decltype(mc)::value;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = sums_by(m - 1); i < sums_by(m); ++i) {
      if ((i & 15) == 0) {
        psum[i >> 4] = e[i];
      } else {
        psum[i >> 4] += e[i];
        pin(psum[i >> 4]);
      }
    }
#pragma unroll
    for (int i = m ? args_by(m - 1) : 0; i < args_by(m); ++i) {
      t[i] = __builtin_fmaf(w.s[kSet][i >> 4][i & 15], scale_log2, -w.m[i >> 4]);
      pin(t[i]);
    }
#pragma unroll
    for (int i = exps_by(m - 1); i < exps_by(m); ++i) {
      e[i] = fast_exp2(t[i]);
      pin(e[i]);
    }
#pragma unroll
    for (int i = packs_by(m - 1); i < packs_by(m); ++i) {
      uint32_t x;
      pack_to(x, e[2 * i], e[2 * i + 1]);
      w.p[kSet][i >> 3][(i & 7) >> 2][i & 3] = x;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // loads n and n + 1 (0 .. 7 of K, 8 .. 15 of V)
  auto copy = [&](auto nc) __attribute__((always_inline)) {
    constexpr int n = decltype(nc)::value;
    if constexpr (n < 8 && kHk >= 0) copy_2k<kHk * kHalfBytes + n * 1024>(cp.k, la.voffK[kHk * 8 + n], la.voffK[kHk * 8 + n + 1], cp.lds);
    if constexpr (n >= 8 && kHv >= 0) copy_2k<kVAt + kHv * kHalfBytes + (n - 8) * 1024>(cp.v, la.voffV[kHv * 8 + n - 8], la.voffV[kHv * 8 + n - 7], cp.lds);
  };
  // fragments of pair f (8 and on: of the next step)
  auto read_v = [&](int f, int a, int vat) __attribute__((always_inline)) {
    if (vat >= 0)
      w.vf[f & 7][a] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) i16x4*)(lds + kVAt + la.vaddr[f & 3][a] + vat + ((f & 7) >> 2) * 4096));
  };
  auto read_k = [&](int f, int kat) __attribute__((always_inline)) {
    if (kat >= 0) w.kf[f & 7] = *reinterpret_cast<const bf16x8*>(lds + la.kaddr[f & 7] + kat);
  };
  auto qk = [&](int f, int g) __attribute__((always_inline)) {
    if (!kQK) return;
    if (f == 0) mfma_first(w.s[kSet ^ 1][g], w.kf[f], q[g][f]);
    else mfma_score(w.s[kSet ^ 1][g], w.kf[f], q[g][f]);
  };
  auto pv = [&](int f, int g) __attribute__((always_inline)) {
    if (kPV) mfma_out(w.o[g][f & 3], join(w.vf[f][0], w.vf[f][1]), w.p[kSet ^ 1][g][f >> 2]);
  };
  auto pair = [&](auto fc) __attribute__((always_inline)) {
    constexpr int f = decltype(fc)::value;
    constexpr int kat = f + kAhead < 8 ? (kQK ? kK : -1) : kKn, vat = f + kAhead < 8 ? (kPV ? kV : -1) : kVn;
    __builtin_amdgcn_sched_barrier(0);
    if (kBar && f + kAhead == 8) asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    qk(f, 0);
    read_v(f + kAhead, 0, vat);
    softmax(std::integral_constant<int, 4 * f>());
    pv(f, 0);
    read_v(f + kAhead, 1, vat);
    if constexpr (f < 2) copy(std::integral_constant<int, 4 * f>());
    softmax(std::integral_constant<int, 4 * f + 1>());
    qk(f, 1);
    read_k(f + kAhead, kat);
    softmax(std::integral_constant<int, 4 * f + 2>());
    pv(f, 1);
    if constexpr (f < 6) copy(std::integral_constant<int, f < 2 ? 4 * f + 2 : 4 + 2 * f>());
    softmax(std::integral_constant<int, 4 * f + 3>());
  };
  pair(std::integral_constant<int, 0>());
  pair(std::integral_constant<int, 1>());
  pair(std::integral_constant<int, 2>());
  pair(std::integral_constant<int, 3>());
  pair(std::integral_constant<int, 4>());
  pair(std::integral_constant<int, 5>());
  pair(std::integral_constant<int, 6>());
  // the last pair: all of the output's MFMAs ahead of what the sums decide
  __builtin_amdgcn_sched_barrier(0);
  pv(7, 0);
  read_v(7 + kAhead, 0, kVn);
  softmax(std::integral_constant<int, 28>());
  pv(7, 1);
  read_v(7 + kAhead, 1, kVn);
  read_k(7 + kAhead, kKn);
  // A lane's sum beyond kOutgrown (infinite for the first keys that a row sees, against the initial maximum) says that one of
  // its two rows may have outgrown its reference maximum; which, each row's 16 tell.  The scores are still there: the step's
  // softmax is done again.  That costs one compare instead of 16 maxima and an exchange per row group.
  __builtin_amdgcn_sched_barrier(0);
  uint64_t outgrown = __ballot(!(psum[0] + psum[1] <= kOutgrown));
  asm volatile("" : "+s"(outgrown));
  __builtin_amdgcn_sched_barrier(0);
  qk(7, 0);                                        // (of the next step's scores: what is done again does not touch them)
  __builtin_amdgcn_sched_barrier(0);
  if (__builtin_expect(outgrown != 0, 0)) {
    settle(w.s[kSet][0], w.s[kSet][1]);
    settle(w.o);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      if (!__any(!(psum[g] <= kOutgrown))) continue;
      asm volatile("" : "+v"(w.s[kSet][g]));     // (or its maxima are taken ahead of the branch)
      softmax_slow(w, kSet, g, scale_log2, psum[g]);
    }
    settle();
  }
  w.l[0] += psum[0];
  w.l[1] += psum[1];
  __builtin_amdgcn_sched_barrier(0);
  // (every fragment of the present halves has arrived: those of pair 7 were the last to be requested)
  if (kFree) asm volatile("s_barrier" ::: "memory");
  qk(7, 1);
}

// kHasList = false visits every visible block, the dense baseline (its own symbol, so profiles tell the two apart);
// kPlanned: long lists are cut (attn_plan.h)
template <bool kHasList, bool kPlanned>
__global__ __launch_bounds__(128, 1) void block_sparse_fwd64_kernel(AttnParams) {
  __shared__ __attribute__((aligned(1024))) char lds[kLdsBytes];
  __shared__ __attribute__((aligned(1024))) char stage[2 * kOutStage];

  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char_ptr)lds + (uint32_t)wave * 8192;   // this wavefront's share of half 0 of K
  // The sweep goes from the end of the list to its start: where attention is local, the blocks nearest the queries set the
  // reference maxima, and little outgrows them.
  auto find = [&](const AttnParams& p, int id, Unit& u) __attribute__((always_inline)) {
    if (!find_unit<kHasList, kPlanned, true>(p, id, u) || !find_list<kHasList, kPlanned>(p, u)) return false;
    u.kb = u.kb_next = 0;
    if (u.n_blocks > 0) {
      u.kb = kHasList ? clamp_block(u.list[u.n_blocks - 1], p.nkb) : u.first + u.n_blocks - 1;
      u.kb_next = u.n_blocks > 1 ? (kHasList ? clamp_block(u.list[u.n_blocks - 2], p.nkb) : u.kb - 1) : u.kb;
    }
    u = uniform(u);
    return true;
  };
  // The q-block is copied row-wise (full lines) like a tile, this wavefront's 64 rows to its own shares of V's halves, and K_0
  // to its place.
  auto request = [&](const AttnParams& p, const Unit& u) __attribute__((always_inline)) {
    if (u.n_blocks == 0) return;
    int lane = (int)threadIdx.x;
    asm volatile("" : "+v"(lane));
    lane &= 63;
    const uint32_t q_row = (uint32_t)p.q_sn * 2, k_row = (uint32_t)p.k_sn * 2, last_rows = (uint32_t)(p.Lk - (p.nkb - 1) * kBlk);
    const u32x4 qr = block_resource(p.q + (int64_t)u.head * p.q_sh, q_row * kBlk, q_row * (uint32_t)(p.Lq - (p.nqb - 1) * kBlk), u.qb, p.nqb);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      copy_1k(qr, load_lane(q_row, lane, i & 3) + ((uint32_t)wave * 64 + 4 * i) * q_row, lds0 + (uint32_t)(kVAt + (i >> 3) * kHalfBytes + (i & 7) * 1024));
    const u32x4 kr = block_resource(p.k + (int64_t)u.kvh * p.k_sh, k_row * kBlk, k_row * last_rows, u.kb, p.nkb);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      copy_1k(kr, load_lane(k_row, lane, i & 3) + ((uint32_t)wave * 32 + (uint32_t)((i >> 3) * 64 + 4 * (i & 7))) * k_row,
              lds0 + (uint32_t)((i >> 3) * kHalfBytes + (i & 7) * 1024));
  };

  Unit u;
  {
    const AttnParams& p = reread_params();
    if (p.lists_decide && p.totals) {          // mostly no q-block is this kernel's, or many are
      bool any = false;
      for (int qb = p.qb_begin + (int)(threadIdx.x & 63); qb < p.qb_end; qb += 64) any = any || long_lists(p, (int)p.totals[32 * (qb - p.idx_row0)], (int)p.totals[32 * (qb - p.idx_row0) + 1]);
      if (!__any(any)) return;
    }
    if (!find(p, (int)blockIdx.x, u)) {
      if (!p.queue) return;
      const int id = hand_out<kHasList, kPlanned>(p, threadIdx.x == 0 ? ask_next(p) : 0, wave, (int)threadIdx.x & 63, true, stage);
      if (id < 0) return;
      find(p, id, u);
    }
    request(p, u);
  }
  for (;;) {
    const AttnParams& p = reread_params();
    u = uniform(u);
    int tid = (int)threadIdx.x;
    asm volatile("" : "+v"(tid));        // (what is computed from it is not kept from unit to unit)
    const int lane = tid & 63, r = lane & 31, hh = lane >> 5;
    const __bf16* const kbase = p.k + (int64_t)u.kvh * p.k_sh;
    const __bf16* const vbase = p.v + (int64_t)u.kvh * p.v_sh;
    const int q_pos = u.qb * kBlk + wave * 64 + r + p.kv_off;   // position of this lane's first query token on the key axis
    const int n_blocks = u.n_blocks;
    int kb = u.kb, kb_next = u.kb_next, ticket = 0;
    LaneAddr la;
    frag_addressing(lane, la);
    tile_loads((uint32_t)p.k_sn * 2, lane, wave, la.voffK);
    tile_loads((uint32_t)p.v_sn * 2, lane, wave, la.voffV);

    SweepState w;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      w.m[g] = kNoKey;
      w.l[g] = 0.f;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) w.o[g][dt][v] = 0.f;
    }
    // list entries from the j-th of the sweep on, 64 at a time, a lane each
    int ids = 0;
    auto fetch_ids = [&](int j) {
      int at = n_blocks - 1 - j - lane;
      at = at > 0 ? at : 0;
      ids = clamp_block(p.col_idx[(u.list - (const_i32_ptr)(uintptr_t)p.col_idx) + at], p.nkb);
    };
    Copies cp;
    cp.lds = lds0;
    const uint32_t k_row = (uint32_t)p.k_sn * 2, v_row = (uint32_t)p.v_sn * 2, last_rows = (uint32_t)(p.Lk - (p.nkb - 1) * kBlk);
    auto aim_k = [&](int b) __attribute__((always_inline)) { cp.k = block_resource(kbase, k_row * kBlk, k_row * last_rows, b, p.nkb); };
    auto aim_v = [&](int b) __attribute__((always_inline)) { cp.v = block_resource(vbase, v_row * kBlk, v_row * last_rows, b, p.nkb); };
    if (n_blocks > 0) {
      aim_v(kb);
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) asm volatile("" : "+a"(w.o[g][dt]));       // (cleared while the loads are on their way)
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");       // the queries and K_0
      bf16x8 q[2][8];   // Q^T fragments stay in registers for the whole sweep
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int s = 0; s < 8; ++s) q[g][s] = *reinterpret_cast<const bf16x8*>(lds + kVAt + g * kHalfBytes + wave * 8192 + la.kaddr[s]);
      auto masked = [&](int b) { return (b * kBlk + kBlk > p.Lk) || (p.causal && b * kBlk + kBlk - 1 > u.qb * kBlk + p.kv_off); };
      auto mask = [&](int set, int key0) __attribute__((always_inline)) {
        settle(w.s[set][0], w.s[set][1]);
#pragma unroll
        for (int g = 0; g < 2; ++g) mask_step(w.s[set][g], key0, hh, q_pos + g * 32, p.Lk, p.causal);
      };
      constexpr int kU = 8192, kH = kHalfBytes;
      if (kHasList && n_blocks > 2) fetch_ids(0);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                  // V may take the place of the queries
      const bool mask_first = masked(kb);
      // The scores of the first 32 keys, from which the rows' reference maxima are taken, while the first half of V is
      // requested.  Of the block that the queries stand in, also of the 32 keys they stand among: the more often the largest
      // probability of a row is a power of two, the less rounding it to bf16 costs, and of text the largest is mostly near the
      // query (error of the output 1.64e-3 with these keys, 2.15e-3 without).
      auto copy_v = [&](int i) __attribute__((always_inline)) { copy_1k(cp.v, la.voffV[i] + (i & 1) * 1024, lds0 + (uint32_t)(kVAt + i * 1024)); };
      bf16x8 kf[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) kf[s] = *reinterpret_cast<const bf16x8*>(lds + la.kaddr[s]);
      if (p.causal && mask_first) {
        int sub[2];
        bf16x8 own[2][8];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          sub[g] = (u.qb * kBlk + wave * 64 + g * 32 + 31 + p.kv_off - kb * kBlk) >> 5;
          sub[g] = sub[g] < 0 ? 0 : sub[g];
          sub[g] = sub[g] > 3 ? 3 : sub[g];
#pragma unroll
          for (int s = 0; s < 8; ++s) own[g][s] = *reinterpret_cast<const bf16x8*>(lds + sub[g] * kU + la.kaddr[s]);
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            __builtin_amdgcn_sched_barrier(0);
            if (s == 0) mfma_first(w.s[1][g], own[g][s], q[g][s]);
            else mfma_score(w.s[1][g], own[g][s], q[g][s]);
            if (s == 0) mfma_first(w.s[0][g], kf[s], q[g][s]);
            else mfma_score(w.s[0][g], kf[s], q[g][s]);
            if (g == 0) copy_v(s);
          }
        }
        settle(w.s[1][0], w.s[1][1]);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          mask_step(w.s[1][g], kb * kBlk + sub[g] * 32, hh, q_pos + g * 32, p.Lk, p.causal);
#pragma unroll
          for (int v = 0; v < 16; ++v) w.m[g] = fmaxf(w.m[g], w.s[1][g][v]);
        }
      } else {
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            if (s == 0) mfma_first(w.s[0][g], kf[s], q[g][s]);
            else mfma_score(w.s[0][g], kf[s], q[g][s]);
          }
          copy_v(s);
        }
      }
      bool mask_now = mask_first;
#pragma unroll
      for (int f = 0; f < kAhead; ++f) w.kf[f] = *reinterpret_cast<const bf16x8*>(lds + la.kaddr[f] + kU);
      settle(w.s[0][0], w.s[0][1]);
      if (mask_now) mask(0, kb * kBlk);
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        float mx = w.m[g];
#pragma unroll
        for (int v = 0; v < 16; ++v) mx = fmaxf(mx, w.s[0][g][v]);
        mx = half_max(mx);
        w.m[g] = mx > kNoKey ? mx * p.scale_log2 : kNoKey;
      }
      aim_k(kb_next);
      sweep_step<0, kU, 0, kH, 0, true, false, true, true, -1, -1>(w, q, lds, la, p.scale_log2, cp);
      int j = 0;
      for (; j + 1 < n_blocks; ++j) {
        if (mask_now) mask(1, kb * kBlk + 32);
        sweep_step<1, kH, 0, kH + kU, kU, true, true, false, false, 0, 1>(w, q, lds, la, p.scale_log2, cp);
        if (mask_now) mask(0, kb * kBlk + 64);
        sweep_step<0, kH + kU, kU, 0, kH, true, true, true, true, -1, -1>(w, q, lds, la, p.scale_log2, cp);
        if (mask_now) mask(1, kb * kBlk + 96);
        aim_v(kb_next);
        sweep_step<1, 0, kH, kU, kH + kU, true, true, false, false, 1, 0>(w, q, lds, la, p.scale_log2, cp);
        kb = kb_next;
        mask_now = masked(kb);
        if (mask_now) mask(0, kb * kBlk);
        if (kHasList && ((j + 2) & 63) == 0) fetch_ids(j + 2);
        kb_next = j + 2 < n_blocks ? (kHasList ? __builtin_amdgcn_readlane(ids, (j + 2) & 63) : kb - 1) : kb;
        aim_k(kb_next);
        sweep_step<0, kU, kH + kU, kH, 0, true, true, true, true, -1, -1>(w, q, lds, la, p.scale_log2, cp);
      }
      // the last block (the answer takes 1 to 2 us)
      if (tid == 0 && p.queue) ticket = ask_next(p);
      if (mask_now) mask(1, kb * kBlk + 32);
      sweep_step<1, kH, 0, kH + kU, kU, true, true, false, false, -1, 1>(w, q, lds, la, p.scale_log2, cp);
      if (mask_now) mask(0, kb * kBlk + 64);
      sweep_step<0, kH + kU, kU, -1, kH, true, true, true, false, -1, -1>(w, q, lds, la, p.scale_log2, cp);
      if (mask_now) mask(1, kb * kBlk + 96);
      sweep_step<1, 0, kH, -1, kH + kU, false, true, false, false, -1, -1>(w, q, lds, la, p.scale_log2, cp);
#pragma unroll
      for (int f = 0; f < 8; ++f) {
#pragma unroll
        for (int g = 0; g < 2; ++g) mfma_out(w.o[g][f & 3], join(w.vf[f][0], w.vf[f][1]), w.p[1][g][f >> 2]);
        if (f + kAhead < 8) {
#pragma unroll
          for (int a = 0; a < 2; ++a)
            w.vf[f + kAhead][a] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) i16x4*)(lds + kVAt + la.vaddr[(f + kAhead) & 3][a] + kH + kU + ((f + kAhead) >> 2) * 4096));
        }
      }
      settle(w.o);
      asm volatile("s_barrier" ::: "memory");      // both wavefronts are done with the tiles
    } else {
      if (tid == 0 && p.queue) ticket = ask_next(p);
    }
    // the last barrier of the sweep left the tiles unused: the next unit's queries and K_0 are on their way while the results leave
    Unit n = u;
    int id = -1;
    if (p.queue) {
      const AttnParams& p = reread_params();
      id = hand_out<kHasList, kPlanned>(p, ticket, wave, lane, n_blocks < 16, stage);
      if (id >= 0) {
        find(p, id, n);
        request(p, n);
      }
    }
    bool whole = true;
    if (kPlanned && u.cuts > 0) {
      float* const part = p.plan.part + (int64_t)u.part0 * kPartFloats;
#pragma unroll
      for (int g = 0; g < 2; ++g) store_partial(part + (int64_t)u.piece * kPartFloats, wave * 2 + g, lane, r, hh, w.o[g], w.m[g], w.l[g]);
      wait_vm0();                              // written through to memory
      __syncthreads();
      int* const scratch = reinterpret_cast<int*>(stage);
      if (tid == 0) scratch[0] = __hip_atomic_fetch_add(p.plan.done + unit_slot(p, u), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      whole = __builtin_amdgcn_readfirstlane(scratch[0]) == u.cuts - 1;      // the piece that comes last combines them
      __syncthreads();
      if (whole) {
#pragma unroll
        for (int g = 0; g < 2; ++g) load_partials(part, u.cuts, wave * 2 + g, lane, r, hh, w.o[g], w.l[g]);
      }
    }
    if (whole) {
#pragma unroll
      for (int g = 0; g < 2; ++g) store_out(p, u.head, u.qb, wave * 2 + g, lane, r, hh, w.o[g], w.l[g], stage + wave * kOutStage);
    }
    if (id < 0) return;
    u = n;
  }
}

}  // namespace xattn
