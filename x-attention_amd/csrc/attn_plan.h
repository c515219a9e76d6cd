// How long lists of the block-sparse attention are shared among workgroups.
//
// A workgroup works through its list one 128-key block after the other, 1.7 to 3.5 us each, and the longest list bounds
// the launch: a chunk on top of a cache has few (head, q-block) units (32 .. 2000) and lists of up to hundreds of blocks,
// and some heads of a prompt keep a hundred times as many blocks as others.  So long lists are cut into pieces, equal in
// length but for the last - where the heads of their q-block differ or units are few (piece_blocks): where every list is as
// long as the next, cutting takes nothing off the end of the launch.
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
constexpr int kPartFloats = 128 * 128 + 2 * 128;   // of one piece: outputs (accumulator order), row maxima, row sums
constexpr int kMostPieces = 16;                    // of a list: the one that comes last combines them alone

// What does not depend on the lists.
struct PlanShape {
  int per_qb;                 // pieces that the lists of one q-block may have together; 0: nothing is cut
  int spread;                 // a q-block of unlike lists is cut for so many pieces in the whole problem
  int min_piece;              // blocks of the shortest piece
  int units;                  // lists of the whole problem, heads x q-blocks
  int nqb;
  int in_turn;                // pieces go to the XCDs in turn
  int rests_last;             // rests go behind the other pieces (PieceIds)
  int last, last_pieces;      // the problem's last q-block, if rows are missing from it (else -1), and its share
};

struct AttnPlan {
  // kNotedStep words apart: pieces noted, of their list's piece length (32 bits) and rests (32); then, per q-block, its lists that are
  // made (16 bits), those of them longer than min_piece (16) and the blocks of all (32).  Set to zero, with `cut` behind it, before
  // lists are noted
  unsigned long long* noted;
  uint32_t* cut;              // [lists] of a list longer than min_piece: its length, until its q-block is noted, then its pieces
                              // (cut_word), or 0 if it stays whole
  int32_t* done;              // [lists] pieces of a cut list that are finished
  int32_t* pieces;            // [room][2] unit, index of the piece in its list: from the front those of their list's piece length, from the
                              // end the rests
  float* part;                // [the same][kPartFloats]
  int room;                   // plan_pieces()
  PlanShape shape;
};

// Ids of the pieces noted: a multiple of 8 of the long ones, behind them of the rests.  The launch deals ids in order, so the
// rests, of half a piece on average, fill up the last round: with them among the others the end of a launch was a piece of full
// length wide (2048 tokens on 63488: the last 80 of 336 us with half of the places empty).  With that, and what stays whole dealt
// to the XCDs in turn (find_place), calls, us: 2048 on 63488 361 -> 347, on 20000 217 -> 204, 1000 on 30000 182 -> 173, 5000 on 30000
// 584 -> 563, 700 of 28 / 4 heads on 20000 111 -> 106, 3000 of 32 / 32 on 20000 405 -> 397; 500 on 60000, 8000 on 100000 and 2048 of
// 32 / 32 on 63488 equal.  Only on a cache: behind a prompt's pieces its many units fill the end, 4096 tokens of 32 / 32
// 77.7 -> 78.6, 9000 182 -> 183.5, 12000 of 32 / 8 215 -> 216.5.
struct PieceIds {
  int whole, rests;           // pieces
  __host__ __device__ int whole_ids() const { return (whole + 7) / 8 * 8; }
  __host__ __device__ int ids() const { return whole_ids() + (rests + 7) / 8 * 8; }
};
// ... of which a launch has room for so many.
inline int64_t piece_ids_room(int64_t pieces) { return pieces ? (pieces + 14) / 8 * 8 : 0; }

// The 512 workgroup slots get about four pieces each (the problem taken to be like the q-block), fewer of which even out
// less: 2048 tokens on 63488 806 us with up to 8192 pieces, 884 with 2048, 977 with 1024.  Of a prompt by itself, whose
// units are many, two each up to 2048 units.  A quarter on top is for the pieces that rounding adds.  A last q-block that
// lacks rows (see piece_blocks) may have 512.  A plan so takes up to 120 or 200 MB, and its launch has up to 1792 or 3072
// workgroups beside the units, 1 to 2 us per thousand where they are spare.
// Not cut: 16 key blocks or fewer, which make short lists; more than 4096 units of a prompt or 8192 on top of a cache at
// least as long as the chunk (a prompt of 32768 tokens 2158 us uncut, 2781 in two: partial results and the spread of a KV
// head over the chip cost more than the end of a long launch).
// A piece costs about 7 us beside its blocks (first tiles, partial result, its part of the combination), so it is not made
// short where lists are long; where keys are few the longest list still bounds the launch.  Whole calls with pieces of at
// least 8 / 16 blocks, us, seeds with long lists: 2048 tokens on 63488 274, 487, 849 / 274, 446, 771; 500 on 60000
// 195, 283 / 181, 250; a prompt of 8000 tokens 235 / 214, of 4096 91 / 100, of 2500 67 / 76.
// Pieces are noted q-block after q-block.  An XCD gets a run of them, adjacent q-blocks over the same keys - but of a long
// prompt's, whose last q-blocks have pieces several times as long as the first, each XCD gets every eighth (runs / in turn, us:
// prompts of 8000 tokens 211 / 218, 12000 430 / 392, 16000 664 / 609; 2048 on 63488 411 / 463, 1000 on 30000 219 / 248).
inline PlanShape plan_shape(int heads, int q_len, int k_len) {
  PlanShape s{};
  const int nqb = (int)(((int64_t)q_len + 127) / 128), nkb = (int)(((int64_t)k_len + 127) / 128);
  const int64_t units = (int64_t)heads * nqb;
  const bool cached = nkb >= 2 * nqb;
  if (nkb <= 16 || units > (cached ? 8192 : 4096)) return s;
  s.spread = cached || units > 2048 ? 2048 : 1024;
  s.min_piece = nkb >= 48 ? 16 : 8;
  s.units = (int)units;
  s.nqb = nqb;
  s.in_turn = !cached && units > 2048;
  s.rests_last = cached;
  const int64_t a_list = (nkb + s.min_piece - 1) / s.min_piece, most = heads * (a_list < kMostPieces ? a_list : kMostPieces);
  const int64_t share = s.spread * 5 / 4 / nqb;
  s.per_qb = (int)(share < most ? share : most);
  if (s.per_qb < 2) s.per_qb = 0;
  s.last = q_len % 128 ? nqb - 1 : -1;
  s.last_pieces = (int)(most < 512 ? most : 512);
  if (s.last_pieces < s.per_qb) s.last_pieces = s.per_qb;
  return s;
}

// Bytes of a plan for a launch of `q_blocks` q-blocks, with `lists` lists in memory, and the plan laid out there (256-byte
// aligned).
inline size_t plan_round(size_t x) { return (x + 255) & ~(size_t)255; }
inline size_t plan_noted_bytes(int nqb) { return plan_round((size_t)(nqb + 1) * kNotedStep * 8); }
inline size_t plan_pieces(const PlanShape& s, int q_blocks) { return (size_t)q_blocks * s.per_qb + (s.last >= 0 ? s.last_pieces - s.per_qb : 0); }
inline size_t plan_bytes(const PlanShape& s, int64_t lists, int q_blocks) {
  if (s.per_qb == 0) return 0;
  const size_t pieces = plan_pieces(s, q_blocks);
  return plan_noted_bytes(s.nqb) + 2 * plan_round((size_t)lists * 4) + plan_round(pieces * 8) + pieces * kPartFloats * sizeof(float);
}
inline AttnPlan plan_at(const PlanShape& s, char* at, int64_t lists, int q_blocks) {
  AttnPlan p{};
  p.shape = s;
  if (s.per_qb == 0) return p;
  p.noted = reinterpret_cast<unsigned long long*>(at);
  p.room = (int)plan_pieces(s, q_blocks);
  p.cut = reinterpret_cast<uint32_t*>(at += plan_noted_bytes(s.nqb));
  p.done = reinterpret_cast<int32_t*>(at += plan_round((size_t)lists * 4));
  p.pieces = reinterpret_cast<int32_t*>(at += plan_round((size_t)lists * 4));
  p.part = reinterpret_cast<float*>(at + plan_round(plan_pieces(s, q_blocks) * 8));
  return p;
}

// Units beyond which lists that are all alike stay whole: cut in three they would take more than two rounds of the 512
// workgroup slots.
constexpr int kEvenUnits = 341;

// Blocks of a piece of the lists of q-block qb - `heads` of them with `total` blocks, the longest with `longest` - or 0: they
// stay whole.  Where the last q-block lacks rows, its estimate is flat and the lists of all its heads are long, whatever the
// others' are: 228 blocks against 6 for 1554 tokens on 37213.  These always are cut.  Otherwise, of text whose heads keep unlike lists the longest is 2 to 5 times the mean, of video, fields, diffuse text
// and dense attention 1.0 to 1.25 times; these are cut where units leave slots idle (into three: long ones only).
// Whole calls, us, not cut / cut whatever the lists: uneven text, 2048 tokens on 63488 1346 / 806, 4096 on 100000
// 2283 / 1397, a prompt of 8000 248 / 211; video of 4096 tokens 135 / 152, of 18000 1432 / 1906; a field of 4096 230 / 297;
// diffuse text of 16000 1654 / 2251; dense 2100 49 / 63, 16384 2008 / 2475; dense 500 on 8700 (128 units) 153 / 115; in
// three with 512 units, dense 2048 on 16000 525 / 587, diffuse text 2048 on 63488 1700 / 1885.
__host__ __device__ inline int piece_blocks(const PlanShape& s, int qb, int heads, int total, int longest) {
  if (longest <= s.min_piece) return 0;
  if (qb == s.last) return s.min_piece;
  int64_t n;
  if (2 * (int64_t)longest * heads >= 3 * (int64_t)total)
    n = ((int64_t)total * s.nqb + s.spread - 1) / s.spread;
  else if (s.units <= 256)
    n = ((int64_t)total * s.nqb + 1023) / 1024;
  else if (s.units <= kEvenUnits && longest >= 64)
    n = (longest + 2) / 3;
  else
    return 0;
  return n > s.min_piece ? (int)(n < 1 << 28 ? n : 1 << 28) : s.min_piece;
}
// Pieces of a list of `count` blocks, and their length, where a q-block's have `blocks`; 0: it is not cut (or too long for
// cut_word: over 30 million keys)
__host__ __device__ inline int list_piece(int count, int blocks) {
  const int n = (int)(((uint32_t)count + kMostPieces - 1) / kMostPieces);
  return n > blocks ? n : blocks;
}
__host__ __device__ inline int list_pieces(int count, int blocks) {
  if (blocks == 0 || count <= blocks || list_piece(count, blocks) >= 1 << 14) return 0;
  return (int)((uint32_t)(count - 1) / (uint32_t)list_piece(count, blocks)) + 1;
}
// The blocks of a q-block's pieces, given what its lists' pieces of a length add up to: twice as many, and again, if they are
// more than its share.  (A list of n > b blocks has less than n / b + 1 < 2 n / b pieces of b, so of twice the b that piece_blocks
// gave an ordinary q-block they are less than total / b, which is within its share.)
template <typename F>
__host__ __device__ inline int fitting_blocks(const PlanShape& s, int qb, int heads, int total, int longest, F pieces_of) {
  int blocks = piece_blocks(s, qb, heads, total, longest);
  while (pieces_of(blocks) > (qb == s.last ? s.last_pieces : s.per_qb)) blocks *= 2;      // (none once no list is longer)
  return blocks;
}

// Where the first piece of a list stands among all pieces (less than 2^14), how many there are (2 .. 16) and the length of all
// but the last (less than 2^14).
__host__ __device__ inline uint32_t cut_word(int at, int pieces, int length) { return (uint32_t)at << 18 | (uint32_t)(pieces - 1) << 14 | (uint32_t)length; }
__host__ __device__ inline int cut_at(uint32_t w) { return (int)(w >> 18); }
__host__ __device__ inline int cut_pieces(uint32_t w) { return (int)(w >> 14 & 15) + 1; }
__host__ __device__ inline int cut_length(uint32_t w) { return (int)(w & 16383); }

// Pieces 0 .. pieces - 1 of a list, each read while the one before it is added: request(x, s) has piece s on its way to x, one
// of a and b.  None beyond the last is requested.
template <typename X, typename R, typename A>
__host__ __device__ __forceinline__ void read_ahead(int pieces, X& a, X& b, R request, A add) {
  request(a, 0);
  int s = 0;
  for (; s + 2 < pieces; s += 2) {
    request(b, s + 1);
    add(a);
    request(a, s + 2);
    add(b);
  }
  if (s + 1 < pieces) {
    request(b, s + 1);
    add(a);
    add(b);
  } else {
    add(a);
  }
}

// Notes the lists of q-block qb, `total` blocks in all, by a whole wavefront: count(h) is the length of head h's where it
// is longer than min_piece, unit0 + h * unit_step its place; reserve(x), called by one lane, adds x to what is noted of pieces and
// gives what was.
template <typename F, typename R>
__device__ __forceinline__ void note_q_block(const AttnPlan& p, int qb, int heads, int total, int unit0, int unit_step, int lane, F count, R reserve) {
  const int first = lane < heads ? count(lane) : 0;
  auto length = [&](int h) { return h < 64 ? first : count(h); };
  int longest = 0;
  for (int h = lane; h < heads; h += 64) longest = length(h) > longest ? length(h) : longest;
  longest = (int)wave_max((uint32_t)longest);
  if (longest <= p.shape.min_piece) return;
  int mine = 0, upto = 0;
  const int blocks = fitting_blocks(p.shape, qb, heads, total, longest, [&](int b) {
    mine = 0;
    for (int h = lane; h < heads; h += 64) mine += list_pieces(length(h), b);
    upto = wave_scan(mine);
    return __builtin_amdgcn_readlane(upto, 63);
  });
  const int sum = blocks ? __builtin_amdgcn_readlane(upto, 63) : 0;
  auto has_rest = [&](int len, int n) { return n && p.shape.rests_last && len < n * list_piece(len, blocks) ? 1 : 0; };
  int my_rests = 0, rests_upto = 0;
  if (p.shape.rests_last) {
    for (int h = lane; h < heads; h += 64) my_rests += has_rest(length(h), list_pieces(length(h), blocks));
    rests_upto = wave_scan(my_rests);
  }
  const int rests = __builtin_amdgcn_readlane(rests_upto, 63);
  unsigned long long before = 0;
  if (lane == 63 && sum > 0) before = reserve((unsigned long long)(uint32_t)rests << 32 | (uint32_t)(sum - rests));
  const int whole0 = __builtin_amdgcn_readlane((int)(uint32_t)before, 63), rests0 = __builtin_amdgcn_readlane((int)(uint32_t)(before >> 32), 63);
  int at = whole0 + rests0 + upto - mine, rest = rests0 + rests_upto - my_rests, whole = at - rest;
  for (int h = lane; h < heads; h += 64) {
    const int len = length(h), n = list_pieces(len, blocks), unit = unit0 + h * unit_step;
    if (len <= p.shape.min_piece) continue;
    p.cut[unit] = n ? cut_word(at, n, list_piece(len, blocks)) : 0;
    p.done[unit] = 0;
    for (int i = 0; i < n; ++i) {
      const int to = i == n - 1 && has_rest(len, n) ? p.room - 1 - rest++ : whole++;
      p.pieces[2 * to] = unit;
      p.pieces[2 * to + 1] = i;
    }
    at += n;
  }
}

// A wavefront has made the list of `count` blocks (the same in every lane) of `head` and q-block `row`, one of the `rows` that
// the lists hold per head (all of the problem's).  Whoever brings the last of the q-block's lists notes them all: a long list's
// length has reached memory that every XCD sees before it is counted, short ones are counted only.  That is a wait for one
// atomic (0.5 us of a prompt's 63 where no list is long), and for the last of unlike lists a store, a load and a second atomic
// (the selection of 4096 tokens 14.3 -> 16.4 us, of 2048 on 63488 32 -> 34.5).
__device__ __forceinline__ void list_made(const AttnPlan& p, int heads, int rows, int row, int head, int count, int lane) {
  unsigned long long before = 0;
  const bool is_long = count > p.shape.min_piece;
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
  note_q_block(
      p, row, heads, total, row, rows, lane,
      [&](int h) { return (int)__hip_atomic_load(p.cut + (int64_t)h * rows + row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); },
      [&](unsigned long long x) { return __hip_atomic_fetch_add(p.noted, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); });
}

}  // namespace xattn
