// Host-only check: launches of few q-blocks give all eight XCDs work, none more than twice the mean rounded up, and still
// produce every (head, q-block) once.  Exit status 0 when all hold.  No GPU call is made.
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
  // runs that are even already keep whole units
  const xattn::DispatchShape whole = xattn::dispatch_shape(24, 24, 313), one = xattn::dispatch_shape(24, 24, 40);
  bad += whole.unit_rows != 64 || whole.unit_shift != 6 || one.unit_rows != 40;
  return bad ? 1 : 0;
}
