// Host-only check of the weights that CUs without a tile pull (proj_pull.h): the pullers of each XCD cover every row of its tiles'
// heads and every step from `ahead` on exactly once, and nothing outside the three weight matrices; and there are pullers only where
// they keep up with the tiles.  Exit status 0 when all hold.  No GPU call is made.
#include <cstdio>
#include <vector>

#include "proj_pull.h"

int main() {
  int bad = 0;
  const int heads[][3] = {{8, 8, 8}, {32, 8, 8}, {28, 4, 4}, {40, 8, 8}, {5, 3, 3}, {3, 1, 1}, {1, 1, 1}, {32, 0, 0}, {40, 0, 0}, {7, 0, 0}, {96, 8, 8}, {64, 8, 8}};
  const int tile[][3] = {{64, 64, 512}, {128, 64, 256}, {128, 128, 256}, {128, 192, 256}, {128, 256, 256}};   // features, tokens, threads
  long launches = 0, pulled = 0;
  for (const auto& h : heads)
    for (const auto& t : tile)
      for (int tokens = 2; tokens <= 1100; tokens += tokens < 140 ? 1 : 37) {
        const int n0 = h[0] * 128, n1 = h[1] * 128, n2 = h[2] * 128;
        const uint32_t mt = (tokens + t[1] - 1) / t[1], total = mt * (uint32_t)((n0 + n1 + n2) / t[0]), per_xcd = (total + 7) / 8;
        if (total > 256) continue;
        ++launches;
        const uint32_t places = xattn::pull_places(tokens, t[1], t[0], total);
        if (!places) continue;
        ++pulled;
        // one workgroup per CU, tiles included; a CU for every tile's features, half of one where several tiles share them
        bool ok = per_xcd + places <= 32 && (mt == 1 ? 4 * places >= 3 * per_xcd : 2 * places * mt >= per_xcd);
        const uint32_t steps = 19, ahead = 3, lanes = places * t[2];
        for (uint32_t x = 0; x < 8 && ok; ++x) {
          std::vector<int> seen((size_t)(n0 + n1 + n2) * steps, 0), want(seen.size(), 0);
          for (uint32_t lane = 0; lane < lanes; ++lane) {
            xattn::PullLane l;
            if (!xattn::pull_lane(x, lane, lanes, per_xcd, total, mt, t[0], n0, n1, ahead, &l)) continue;
            const int n[] = {n0, n1, n2}, from[] = {0, n0, n0 + n1};
            if (l.product < 0 || l.product > 2 || l.row < 0 || l.row >= n[l.product]) { ok = false; break; }
            for (uint32_t s = l.step; s < steps; s += l.every) ++seen[(size_t)(from[l.product] + l.row) * steps + s];
          }
          for (uint32_t lin = x * per_xcd; lin < (x + 1) * per_xcd && lin < total; ++lin)
            for (uint32_t r = lin / mt * t[0] / 128 * 128; r < (lin / mt * t[0] / 128 + 1) * 128; ++r)
              for (uint32_t s = ahead; s < steps; ++s) want[(size_t)r * steps + s] = 1;
          ok = ok && seen == want;
        }
        if (!ok) std::printf("%d + %d + %d heads, %d tokens, tile %d x %d: wrong\n", h[0], h[1], h[2], tokens, t[0], t[1]);
        bad += !ok;
      }
  std::printf("%ld launches, %ld with pullers\n", launches, pulled);
  // too few CUs left over, which would still pull when the tiles are done: 2 tokens of 224 and 160 tiles, 128 of 224, 192 of 240
  const int late[][3] = {{2, 64, 224}, {2, 64, 160}, {128, 64, 224}, {192, 64, 240}, {2, 64, 256}};
  for (const auto& c : late) bad += xattn::pull_places(c[0], c[1], 64, c[2]) != 0;
  // enough of them, with a last token tile that lacks rows or not: tokens, tile (tokens, features), tiles
  const int gain[][4] = {{2, 64, 64, 16}, {64, 64, 64, 96}, {72, 64, 64, 128}, {128, 64, 64, 128}, {200, 64, 128, 160}, {330, 64, 128, 144},
                         {400, 128, 128, 192}, {500, 128, 128, 192}, {1000, 128, 128, 192}, {1400, 192, 128, 192}, {1000, 256, 128, 192}};
  for (const auto& c : gain) bad += xattn::pull_places(c[0], c[1], c[2], c[3]) == 0;
  return bad || pulled == 0 ? 1 : 0;
}
