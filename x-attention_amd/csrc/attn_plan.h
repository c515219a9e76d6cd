// How long lists of the block-sparse attention are shared among workgroups.
//
// A workgroup works through its list one 128-key block after the other, 1.7 to 3.5 us each, and the longest list bounds
// the launch: a chunk on top of a cache has few (head, q-block) units (32 .. 2000) and lists of up to hundreds of blocks,
// and some heads of a prompt keep a hundred times as many blocks as others.  So lists of more than `min_piece` blocks are
// cut into at most `items` pieces, equal in length but for the last - where the heads of their q-block differ or units are
// few (most_pieces): where every list is as long as the next, cutting takes nothing off the end of the launch.
// A q-block's lists are noted by whoever completes the last of them.  The attention launch deals its workgroups first to
// the pieces, then to the units - whose list, if it is cut, is no longer theirs - and those for which nothing is left come
// last, beside the end of the work.  Each piece leaves (output, maximum, sum) unnormalised in fp32, and whichever comes
// last combines them in their order.
//
// Where a list is cut depends on the lengths of its q-block's lists and on the size of the whole problem alone, so results
// do not depend on how a problem is spread over launches.
#pragma once
#include "xattn_common.h"

namespace xattn {

constexpr int kNotedStep = 16;                     // 128 bytes: counters that many wavefronts add to share no line
constexpr int kPartFloats = 128 * 128 + 2 * 128;   // of one item: outputs (accumulator order), row maxima, row sums

struct AttnPlan {
  // kNotedStep words apart: pieces noted; then, per q-block, its lists that are made (16 bits), those of them longer than
  // min_piece (16) and the blocks of all (32).  Set to zero, with `cut` behind it, before lists are noted
  unsigned long long* noted;
  uint32_t* cut;              // [lists] of a list longer than min_piece: its length, until its q-block is noted, then its pieces
                              // (cut_word), or 0 if it stays whole
  int32_t* pieces;            // [units * items][2] unit, index of the piece in its list
  int32_t* done;              // [lists] pieces of a cut list that are finished
  float* part;                // [units * items][kPartFloats]
  int items;                  // most pieces of a list; 0: no plan
  int min_piece;              // blocks of the shortest
  int units;                  // lists of the whole problem
  int in_turn;                // pieces go to the XCDs in turn
};

// Pieces a list may be cut into, for a problem of `units` lists (heads x q-blocks) over nkb key blocks; 1: never.  The
// launch has units * pieces workgroups for them, and where lists are short the spare ones cost 1 - 2 us per thousand: for a
// prompt by itself about 2048 beside the units, and two pieces up to 4096 units (whole calls, us, uneven lists: 4096 tokens
// 125 uncut, 92 cut; 16000 tokens 679 and 497 uncut, 652 and 478 in two; 32768 tokens 2158 uncut, 2781 in two - partial
// results and the spread of a KV head over the chip cost more than the end of a long launch).  On top of a cache at least
// as long as the chunk, where lists are long and few, 8192 (2048 tokens on 63488: 1426 uncut, 881 with 8192, 1005 with 2048;
// 64 on 100000: 1461 and 334; 8000 on 100000: 3865 and 2765).  16 key blocks or fewer make short lists.
inline int plan_items(int64_t units, int nqb, int nkb) {
  const bool cached = nkb >= 2 * nqb;
  if (nkb <= 16 || units > (cached ? 8192 : 4096)) return 1;
  const int64_t n = (cached ? 8192 : 2048) / units + 1;
  return n > 16 ? 16 : n < 2 ? 2 : (int)n;
}
// A piece costs about 7 us beside its blocks (first tiles, partial result, its part of the combination), so it is not made
// short where lists are long; where keys are few the longest list still bounds the launch.  Whole calls with pieces of at
// least 8 / 16 blocks, us, seeds with long lists: 2048 tokens on 63488 274, 487, 849 / 274, 446, 771; 500 on 60000
// 195, 283 / 181, 250; a prompt of 8000 tokens 235 / 214, of 4096 91 / 100, of 2500 67 / 76.
inline int min_piece(int nkb) { return nkb >= 48 ? 16 : 8; }

// Units beyond which lists that are all alike stay whole: cut in three they would take more than two rounds of the 512
// workgroup slots.
constexpr int kEvenUnits = 341;

// Pieces are noted q-block after q-block.  An XCD gets a run of them, adjacent q-blocks over the same keys - but of a long
// prompt's, whose last q-blocks have pieces several times as long as the first, each XCD gets every eighth (runs / in turn, us:
// prompts of 8000 tokens 211 / 218, 12000 430 / 392, 16000 664 / 609; 2048 on 63488 411 / 463, 1000 on 30000 219 / 248).

// Bytes of a plan for `units` of the `lists` lists in memory, of a problem of nqb q-blocks, and the plan laid out there
// (256-byte aligned).
inline size_t plan_round(size_t x) { return (x + 255) & ~(size_t)255; }
inline size_t plan_noted_bytes(int nqb) { return plan_round((size_t)(nqb + 1) * kNotedStep * 8); }
inline size_t plan_bytes(int64_t lists, int64_t units, int nqb, int items) {
  if (items <= 1) return 0;
  return plan_noted_bytes(nqb) + 2 * plan_round((size_t)lists * 4) + plan_round((size_t)units * items * 8) +
         (size_t)units * items * kPartFloats * sizeof(float);
}
inline AttnPlan plan_at(char* at, int64_t lists, int64_t units, int64_t problem_units, int nqb, int nkb, int items) {
  AttnPlan p{};
  if (items <= 1) return p;
  p.items = items;
  p.min_piece = min_piece(nkb);
  p.units = (int)problem_units;
  p.in_turn = nkb < 2 * nqb && problem_units > 2048;
  p.noted = reinterpret_cast<unsigned long long*>(at);
  p.cut = reinterpret_cast<uint32_t*>(at += plan_noted_bytes(nqb));
  p.done = reinterpret_cast<int32_t*>(at += plan_round((size_t)lists * 4));
  p.pieces = reinterpret_cast<int32_t*>(at += plan_round((size_t)lists * 4));
  p.part = reinterpret_cast<float*>(at + plan_round((size_t)units * items * 8));
  return p;
}

// Most pieces of a list of a q-block whose `heads` lists have `total` blocks, the longest of them `longest`; 0: they stay
// whole.  Of text whose heads keep unlike lists the longest is 2 to 5 times the mean, of video, fields, diffuse text and
// dense attention 1.0 to 1.25 times; these are cut where units leave slots idle (into three: long ones only).
// Whole calls, us, not cut / cut whatever the lists: uneven text, 2048 tokens on 63488 1346 / 806, 4096 on 100000
// 2283 / 1397, a prompt of 8000 248 / 211; video of 4096 tokens 135 / 152, of 18000 1432 / 1906; a field of 4096 230 / 297;
// diffuse text of 16000 1654 / 2251; dense 2100 49 / 63, 16384 2008 / 2475; dense 500 on 8700 (128 units) 153 / 115; in
// three with 512 units, dense 2048 on 16000 525 / 587, diffuse text 2048 on 63488 1700 / 1885.
__host__ __device__ inline int most_pieces(const AttnPlan& p, int heads, int total, int longest) {
  if (longest <= p.min_piece) return 0;
  if (2 * (int64_t)longest * heads >= 3 * (int64_t)total || p.units <= 256) return p.items;
  return p.units <= kEvenUnits && longest >= 64 ? 3 : 0;
}
__host__ __device__ inline int piece_length(int count, int most, int min_piece) {
  const int n = (int)(((uint32_t)count + (uint32_t)most - 1) / (uint32_t)most);
  return n > min_piece ? n : min_piece;
}
// pieces of a list of `count` blocks of such a q-block; 0: it is not cut (or too long for cut_word: over 4 million keys)
__host__ __device__ inline int piece_count(int count, int most, int min_piece) {
  if (!most || count <= min_piece || piece_length(count, most, min_piece) >= 1 << 14) return 0;
  return (int)((uint32_t)(count - 1) / (uint32_t)piece_length(count, most, min_piece)) + 1;
}

// Where the first piece of a list stands among all pieces (less than 2^14), how many there are (2 .. 16) and the length of all
// but the last (less than 2^14).
__host__ __device__ inline uint32_t cut_word(int at, int pieces, int length) { return (uint32_t)at << 18 | (uint32_t)(pieces - 1) << 14 | (uint32_t)length; }
__host__ __device__ inline int cut_at(uint32_t w) { return (int)(w >> 18); }
__host__ __device__ inline int cut_pieces(uint32_t w) { return (int)(w >> 14 & 15) + 1; }
__host__ __device__ inline int cut_length(uint32_t w) { return (int)(w & 16383); }

// Notes the lists of one q-block, `total` blocks in all, by a whole wavefront: count(h) is the length of head h's where it
// is longer than min_piece, unit0 + h * unit_step its place.
template <typename F>
__device__ __forceinline__ void note_q_block(const AttnPlan& p, int heads, int total, int unit0, int unit_step, int lane, F count) {
  const int first = lane < heads ? count(lane) : 0;
  auto length = [&](int h) { return h < 64 ? first : count(h); };
  int longest = 0;
  for (int h = lane; h < heads; h += 64) longest = length(h) > longest ? length(h) : longest;
  longest = (int)wave_max((uint32_t)longest);
  if (longest <= p.min_piece) return;
  const int most = most_pieces(p, heads, total, longest);
  int mine = 0;
  for (int h = lane; h < heads; h += 64) mine += piece_count(length(h), most, p.min_piece);
  const int upto = wave_scan(mine);
  int at = 0;
  if (lane == 63 && upto > 0) at = (int)__hip_atomic_fetch_add(p.noted, (unsigned long long)upto, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  at = __builtin_amdgcn_readlane(at, 63) + upto - mine;
  for (int h = lane; h < heads; h += 64) {
    const int len = length(h), n = piece_count(len, most, p.min_piece), unit = unit0 + h * unit_step;
    if (len <= p.min_piece) continue;
    p.cut[unit] = n ? cut_word(at, n, piece_length(len, most, p.min_piece)) : 0;
    p.done[unit] = 0;
    for (int i = 0; i < n; ++i) {
      p.pieces[2 * (at + i)] = unit;
      p.pieces[2 * (at + i) + 1] = i;
    }
    at += n;
  }
}

// A wavefront has made the list of `count` blocks (the same in every lane) of `head` and the q-block in row `row` of the
// `rows` rows that the lists hold per head.  Whoever brings the last of the q-block's lists notes them all: a long list's
// length has reached memory that every XCD sees before it is counted, short ones are counted only (and wait for one atomic:
// 1 to 2 us of a prompt's 60 where no list is long).
__device__ __forceinline__ void list_made(const AttnPlan& p, int heads, int rows, int row, int head, int count, int lane) {
  unsigned long long before = 0;
  const bool is_long = count > p.min_piece;
  if (lane == 0) {
    if (is_long) {
      __hip_atomic_store(p.cut + (int64_t)head * rows + row, (uint32_t)count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    before = __hip_atomic_fetch_add(p.noted + (1 + row) * kNotedStep, (unsigned long long)(uint32_t)count << 32 | (is_long ? 0x10001u : 1u),
                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  asm volatile("" ::: "memory");
  const uint32_t lists = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)before);
  const int total = __builtin_amdgcn_readfirstlane((int)(uint32_t)(before >> 32)) + count;
  if ((lists & 0xffff) != (uint32_t)heads - 1 || (lists >> 16 == 0 && !is_long)) return;
  note_q_block(p, heads, total, row, rows, lane, [&](int h) {
    return (int)__hip_atomic_load(p.cut + (int64_t)h * rows + row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  });
}

}  // namespace xattn
