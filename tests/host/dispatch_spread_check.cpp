// Host-only check of the workgroup map.  At chosen sizes launches of few q-blocks give all eight XCDs work, none more than twice the
// mean rounded up.  At all sizes of up to 130 q-blocks and 26 head layouts every (head, q-block) comes once, the ids of a unit share
// their KV head, and no XCD has more than the fullest of units of 64, and small
// units have no ids without work.  Exit status 0 when all hold.  No GPU call is made.
#include <cstdio>
#include <vector>

#include "attn_tiles.h"

int main() {
  const int cases[][3] = {{28, 4, 8}, {28, 4, 9}, {28, 4, 17}, {8, 2, 16}, {8, 2, 4}, {4, 4, 64}, {4, 4, 2}, {32, 1, 8}, {32, 1, 16},
                          {40, 8, 3}, {12, 12, 40}, {6, 6, 12}, {96, 3, 25}, {24, 24, 313}, {32, 8, 100}, {28, 4, 63}, {28, 4, 72}};
  int bad = 0;
  for (const auto& c : cases) {
    const int H = c[0], Hkv = c[1], n = c[2];
    std::vector<int> seen((size_t)H * n, 0), on(8, 0);
    for (long id = 0; id < (long)xattn::grid_for(H, Hkv, n); ++id) {
      int head, qb;
      if (!xattn::map_workgroup((int)id, H, Hkv, 0, n, &head, &qb)) continue;
      ++seen[(size_t)head * n + qb];
      ++on[id & 7];
    }
    int wrong = 0, most = 0, idle = 0;
    for (int v : seen) wrong += v != 1;
    for (int v : on) most = v > most ? v : most, idle += v == 0;
    const bool ok = wrong == 0 && idle == 0 && most <= 2 * ((H * n + 7) / 8);
    std::printf("H=%d Hkv=%d q-blocks %d: wrong %d idle %d most %d of %d\n", H, Hkv, n, wrong, idle, most, H * n);
    bad += !ok;
  }
  const int layouts[][2] = {{32, 8}, {32, 32}, {28, 4}, {24, 24}, {8, 2}, {16, 2}, {8, 1}, {32, 1}, {64, 4}, {32, 4}, {4, 4}, {12, 12}, {40, 8},
                            {4, 1}, {16, 16}, {7, 1}, {6, 6}, {2, 2}, {1, 1}, {64, 8}, {96, 3}, {14, 2}, {28, 28}, {71, 1}, {20, 4}, {130, 1}};
  for (const auto& l : layouts)
    for (int n = 1; n <= 130; ++n) {
      const int H = l[0], Hkv = l[1], begin = n % 5;
      const xattn::DispatchShape d = xattn::dispatch_shape(H, Hkv, n);
      xattn::DispatchShape whole = d;
      whole.unit_rows = 64 / d.set_heads;
      whole.unit_size = 64;
      whole.unit_inv = 1u << 25;
      std::vector<int> seen((size_t)H * n, 0);
      auto fullest = [&](const xattn::DispatchShape& s, bool check) {
        std::vector<int> on(8, 0);
        int most = 0, wrong = 0;
        for (long id = 0; id < (long)xattn::grid_for(s, n); ++id) {
          int head, qb, kv;
          if (!xattn::map_workgroup((int)id, s, begin, begin + n, &head, &qb, &kv)) continue;
          ++on[id & 7];
          if (!check) continue;
          ++seen[(size_t)head * n + qb - begin];
          int other_head, other_qb, other_kv;                   // the unit's first id has work if any of its has
          const long first = ((id >> 3) / s.unit_size * s.unit_size << 3) + (id & 7);
          wrong += !xattn::map_workgroup((int)first, s, begin, begin + n, &other_head, &other_qb, &other_kv) || other_kv != kv || kv != head / (H / Hkv);
        }
        for (int v : on) most = v > most ? v : most;
        return wrong ? 1 << 30 : most;
      };
      const int now = fullest(d, true), then = fullest(whole, false);
      // where runs are few, units of up to 32 have no ids without work between those with (they would cost their CUs a turn), but for
      // a run that lacks rows
      int gaps = 0;
      if ((n + whole.unit_rows - 1) / whole.unit_rows < 8 && n % d.unit_rows == 0 && d.set_heads * d.unit_rows <= 32)
        for (long id = 0; id < 8L * (d.n_groups * (n / d.unit_rows) / 8) * d.unit_size; ++id) {
          int head, qb, kv;
          gaps += d.sets == 1 && !xattn::map_workgroup((int)id, d, begin, begin + n, &head, &qb, &kv);
        }
      if (gaps) std::printf("H=%d Hkv=%d q-blocks %d: %d ids without work\n", H, Hkv, n, gaps);
      bad += gaps != 0;
      int wrong = 0;
      for (int v : seen) wrong += v != 1;
      if (wrong || now > then) std::printf("H=%d Hkv=%d q-blocks %d: wrong %d, fullest XCD %d, of whole units %d\n", H, Hkv, n, wrong, now, then);
      bad += wrong || now > then;
    }
  // runs that are even already keep whole units
  const xattn::DispatchShape whole = xattn::dispatch_shape(24, 24, 313), one = xattn::dispatch_shape(24, 24, 40);
  bad += whole.unit_rows != 64 || whole.unit_size != 64 || one.unit_rows != 40;
  return bad ? 1 : 0;
}
