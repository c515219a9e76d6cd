// Host-only check of the rule by which the attention kernel's long lists are cut (attn_plan.h), over many problem sizes and
// random lists.  Prints one line per problem size; exit status 0 when all hold.  No GPU call is made.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "attn_plan.h"

using namespace xattn;

int main() {
  std::mt19937 rng(7);
  auto upto = [&](int n) { return (int)(rng() % (uint32_t)(n + 1)); };
  int bad = 0;
  const int cases[][3] = {  // heads, q-blocks, key blocks
      {32, 1, 782}, {32, 4, 72},   {32, 16, 512}, {32, 63, 845}, {32, 256, 1024}, {32, 20, 20},  {32, 32, 32},  {32, 125, 125}, {28, 16, 141},
      {24, 20, 20}, {1, 13, 27},   {1, 3, 4000},  {1, 8000, 16000}, {2, 300, 700}, {72, 12, 33},  {130, 31, 63}, {8, 16, 17},    {4096, 2, 40},
      {3, 3, 43},   {66, 20, 20},  {10, 32, 80},  {11, 31, 64},  {2, 1281, 4000}, {2, 1280, 4000}, {32, 1, 32766}, {1, 1, 300000}, {32, 300, 300},
  };
  for (const auto& c : cases) {
    const int H = c[0], nqb = c[1], nkb = c[2];
    const PlanShape s = plan_shape(H, nqb, nkb);
    const size_t bytes = plan_bytes(s, (int64_t)H * nqb, nqb);
    int cut_lists = 0, whole = 0, faults = bytes > 180000000;
    for (int trial = 0; s.per_qb && trial < 400; ++trial) {
      // even lists, a few long among short ones, anything, half of them long, just above a piece, full
      std::vector<int> n(H);
      const int kind = trial % 6, base = 1 + upto(nkb - 1), longs = 1 + upto(H - 1);
      for (int h = 0; h < H; ++h)
        n[h] = kind == 0 ? std::max(1, base - upto(base / 10)) : kind == 1 ? (h % H < longs / 8 + 1 ? base : 2) : kind == 2 ? upto(nkb)
               : kind == 3 ? (h & 1 ? base : 1) : kind == 4 ? (h < longs ? std::min(nkb, s.min_piece + 1) : 1) : nkb;
      std::shuffle(n.begin(), n.end(), rng);
      int total = 0, longest = 0;
      for (int x : n) total += x, longest = std::max(longest, x);
      auto pieces_of = [&](int b) {
        int sum = 0;
        for (int x : n) sum += list_pieces(x, b);
        return sum;
      };
      const int blocks = fitting_blocks(s, H, total, longest, pieces_of);
      // a q-block that is to be cut fits its share of the pieces
      faults += (blocks == 0) != (piece_blocks(s, H, total, longest) == 0);
      faults += blocks && (pieces_of(blocks) > s.per_qb || blocks < s.min_piece);
      // lists that are all alike stay whole but where units are few
      if (10 * (int64_t)longest * H < 13 * (int64_t)total && H * nqb > kEvenUnits) faults += blocks != 0;
      int at = 0;
      for (int x : n) {
        const int k = list_pieces(x, blocks);
        (k ? cut_lists : whole) += 1;
        if (!k) {
          faults += blocks && x > blocks && list_piece(x, blocks) < 1 << 14;
          continue;
        }
        const uint32_t w = cut_word(at, k, list_piece(x, blocks));
        const int len = cut_length(w);
        faults += w == 0 || cut_at(w) != at || cut_pieces(w) != k || k < 2 || k > kMostPieces;
        faults += (k - 1) * len >= x || k * len < x || len < s.min_piece;
        at += k;
      }
      faults += at > s.per_qb;
    }
    std::printf("H=%d q-blocks %d key blocks %d: per q-block %d, %zu MB, cut %d whole %d, faults %d\n", H, nqb, nkb, s.per_qb, bytes >> 20,
                cut_lists, whole, faults);
    bad += faults != 0;
  }
  return bad ? 1 : 0;
}
