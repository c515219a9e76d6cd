// How long lists of the block-sparse attention are shared among workgroups.
//
// A workgroup works through its list one 128-key block after the other, 1.7 to 3.5 us each, and the longest list bounds
// the launch: a chunk on top of a cache has few (head, q-block) units (32 .. 2000) and lists of up to hundreds of blocks,
// and some heads of a prompt keep a hundred times as many blocks as others.  So lists of more than `min_piece` blocks are
// noted when they are made and cut into at most `items` pieces, equal in length but for the last.  The attention launch
// deals its workgroups first to the pieces, then to the units - whose list, if it is cut, is no longer theirs - and those
// for which nothing is left come last, beside the end of the work.  Each piece leaves (output, maximum, sum) unnormalised in
// fp32, and whichever comes last combines them in their order.
//
// Where a list is cut depends on its length and on the size of the whole problem alone, so results do
// not depend on how a problem is spread over launches.
#pragma once
#include "xattn_common.h"

namespace xattn {

constexpr int kPartFloats = 128 * 128 + 2 * 128;   // of one item: outputs (accumulator order), row maxima, row sums

struct AttnPlan {
  unsigned long long* head;   // low half: pieces noted, high half: lists; set to zero before lists are noted
  int32_t* pieces;            // [units * items][2] unit, index of the piece in its list
  int32_t* number;            // [lists] where a noted list stands among those
  int32_t* done;              // [units] pieces finished, by that number
  float* part;                // [units * items][kPartFloats], a list's own from number * items on
  int items;                  // most pieces of a list; 0: no plan
  int min_piece;              // blocks of the shortest
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

// Bytes of a plan for `units` of the `lists` lists in memory, and the plan laid out there (256-byte aligned).
inline size_t plan_round(size_t x) { return (x + 255) & ~(size_t)255; }
inline size_t plan_bytes(int64_t lists, int64_t units, int items) {
  if (items <= 1) return 0;
  return 256 + plan_round((size_t)units * items * 8) + plan_round((size_t)lists * 4) + plan_round((size_t)units * 4) +
         (size_t)units * items * kPartFloats * sizeof(float);
}
inline AttnPlan plan_at(char* at, int64_t lists, int64_t units, int items, int nkb) {
  AttnPlan p{};
  if (items <= 1) return p;
  p.items = items;
  p.min_piece = min_piece(nkb);
  p.head = reinterpret_cast<unsigned long long*>(at);
  p.pieces = reinterpret_cast<int32_t*>(at += 256);
  p.number = reinterpret_cast<int32_t*>(at += plan_round((size_t)units * items * 8));
  p.done = reinterpret_cast<int32_t*>(at += plan_round((size_t)lists * 4));
  p.part = reinterpret_cast<float*>(at + plan_round((size_t)units * 4));
  return p;
}

__host__ __device__ inline int piece_length(int count, const AttnPlan& p) {
  const int n = (int)(((uint32_t)count + (uint32_t)p.items - 1) / (uint32_t)p.items);
  return n > p.min_piece ? n : p.min_piece;
}
// pieces of a list of `count` blocks, at most items; 0: it is not cut
__host__ __device__ inline int piece_count(int count, const AttnPlan& p) {
  return count > p.min_piece ? (int)((uint32_t)(count - 1) / (uint32_t)piece_length(count, p)) + 1 : 0;
}

// Notes list `unit` of `count` blocks (called by one lane).
__device__ __forceinline__ void note_list(const AttnPlan& p, int unit, int count) {
  const int n = piece_count(count, p);
  if (n == 0) return;
  const unsigned long long old = __hip_atomic_fetch_add(p.head, (1ull << 32) | (unsigned long long)n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int at = (int)(uint32_t)old, number = (int)(old >> 32);
  p.number[unit] = number;
  p.done[number] = 0;
  for (int i = 0; i < n; ++i) {
    p.pieces[2 * (at + i)] = unit;
    p.pieces[2 * (at + i) + 1] = i;
  }
}

}  // namespace xattn
