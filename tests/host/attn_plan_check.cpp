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
  const int cases[][3] = {  // heads, query tokens, key tokens
      {32, 64, 100064},    {32, 500, 9200},     {32, 2048, 65536},   {32, 8000, 108000},  {32, 32768, 131072}, {32, 2500, 2500},
      {32, 4096, 4096},    {32, 16000, 16000},  {28, 2048, 18048},   {24, 2500, 2500},    {1, 1591, 3398},     {1, 300, 512000},
      {1, 1024000, 2048000}, {2, 38400, 89600}, {72, 1500, 4200},    {130, 3900, 8000},   {8, 2048, 2176},     {4096, 130, 5000},
      {3, 300, 5420},      {66, 2500, 2500},    {10, 4096, 10240},   {11, 3968, 8192},    {2, 163900, 512000}, {2, 163840, 512000},
      {32, 128, 4194000},  {1, 1, 38400000},    {32, 38400, 38400},  {28, 1554, 38767},   {32, 6301, 6301},    {600, 129, 4000},
      {32, 4095, 4095},
  };
  for (const auto& c : cases) {
    const int H = c[0], nqb = (c[1] + 127) / 128, nkb = (c[2] + 127) / 128;
    const PlanShape s = plan_shape(H, c[1], c[2]);
    const size_t bytes = plan_bytes(s, (int64_t)H * nqb, nqb);
    size_t most = 0;                       // pieces that the q-blocks may have together
    for (int qb = 0; qb < nqb; ++qb) most += qb == s.last ? s.last_pieces : s.per_qb;
    int cut_lists = 0, whole = 0, faults = bytes > 210000000 || (s.per_qb && most > plan_pieces(s, nqb)) || plan_pieces(s, nqb) >= 1 << 14;
    for (int trial = 0; s.per_qb && trial < 800; ++trial) {
      const int qb = trial % 2 ? nqb - 1 : 0, share = qb == s.last ? s.last_pieces : s.per_qb;
      // even lists, a few long among short ones, anything, half of them long, just above a piece, full
      std::vector<int> n(H);
      const int kind = trial / 2 % 6, base = 1 + upto(nkb - 1), longs = 1 + upto(H - 1);
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
      const int blocks = fitting_blocks(s, qb, H, total, longest, pieces_of);
      // a q-block that is to be cut fits its share of the pieces, an ordinary one with pieces of twice the length at most
      const int first = piece_blocks(s, qb, H, total, longest);
      faults += (blocks == 0) != (first == 0) || (qb != s.last && blocks > 2 * first);
      faults += blocks && (pieces_of(blocks) > share || blocks < s.min_piece);
      // lists that are all alike stay whole but where units are few
      if (10 * (int64_t)longest * H < 13 * (int64_t)total && H * nqb > kEvenUnits && qb != s.last) faults += blocks != 0;
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
      faults += at > share;
    }
    std::printf("H=%d q-blocks %d key blocks %d: per q-block %d, last %d, %zu MB, cut %d whole %d, faults %d\n", H, nqb, nkb, s.per_qb, s.last >= 0 ? s.last_pieces : 0, bytes >> 20,
                cut_lists, whole, faults);
    bad += faults != 0;
  }
  // every piece of a list is added once, in order, and no other is read
  for (int pieces = 1; pieces <= kMostPieces; ++pieces) {
    int a = -1, b = -1, added = 0, faults = 0;
    read_ahead(
        pieces, a, b, [&](int& x, int s) { faults += s < 0 || s >= pieces, x = s; },
        [&](int& x) { faults += x != added++, x = -1; });
    faults += added != pieces;
    std::printf("%d pieces combined, faults %d\n", pieces, faults);
    bad += faults != 0;
  }
  return bad ? 1 : 0;
}
