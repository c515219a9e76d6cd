// Host-only check of the attention kernels' workgroup -> (head, q-block) map:
// over a launch of grid_for() ids every (head, q-block) of the range must be
// produced exactly once and nothing else.  Prints one line per case; exit
// status 0 when all hold.  No GPU call is made.
#include <cstdio>
#include <utility>
#include <vector>

#include "attn_tiles.h"

// every unit once by the map for unlike lists, too
static int unlike_faults(int H, int Hkv, int b, int e) {
  const xattn::DispatchShape d = xattn::unlike_lists_shape(H, Hkv, e - b), whole = xattn::dispatch_shape(H, Hkv, e - b);
  std::vector<int> seen((size_t)H * (e - b), 0);
  int faults = d.unit_rows > whole.unit_rows || d.set_heads * d.unit_rows > (int)d.unit_size;
  for (long id = 0; id < (long)xattn::grid_for(d, e - b); ++id) {
    int head = -1, qb = -1, kv = -1;
    if (!xattn::map_workgroup((int)id, d, b, e, &head, &qb, &kv)) continue;
    if (head < 0 || head >= H || qb < b || qb >= e || kv != head / (H / Hkv)) return 1 << 20;
    ++seen[(size_t)head * (e - b) + (qb - b)];
  }
  for (int v : seen) faults += v != 1;
  // a smaller unit has as many ids as work: what is idle is the rows that its last run lacks and the units that fill up the XCDs
  const int work = d.set_heads * d.unit_rows, runs = (e - b + d.unit_rows - 1) / d.unit_rows;
  if (d.unit_rows < whole.unit_rows) faults += (int)d.unit_size != work || (long)xattn::grid_for(d, e - b) != ((long)runs * d.n_groups + 7) / 8 * 8 * work;
  return faults;
}
// whether units are smaller for unlike lists than for others
static bool smaller(int H, int Hkv, int n) {
  const xattn::DispatchShape d = xattn::unlike_lists_shape(H, Hkv, n), whole = xattn::dispatch_shape(H, Hkv, n);
  return d.unit_rows < whole.unit_rows && d.unit_size < whole.unit_size;
}

int main() {
  for (const auto& l : {std::pair<int, int>{32, 32}, {32, 8}, {28, 4}, {24, 24}, {1, 1}, {7, 1}, {64, 1}, {71, 1}, {96, 3}, {40, 8}, {14, 2}, {12, 12}, {256, 1}})
    for (int n : {1, 40, 47, 48, 49, 63, 64, 65, 100, 127, 133, 255, 256, 257, 313, 512, 931, 1024}) {
      const int faults = unlike_faults(l.first, l.second, n % 5, n % 5 + n);
      if (faults) return std::printf("unlike lists, H=%d Hkv=%d q-blocks %d: faults %d\n", l.first, l.second, n, faults), 1;
    }
  // they are from 48 q-blocks on, while runs are fewer than 16 and units of more than 16
  for (const auto& l : {std::pair<int, int>{32, 32}, {24, 24}, {12, 12}})
    for (int n : {48, 64, 133, 256})
      if (!smaller(l.first, l.second, n)) return std::printf("H=%d Hkv=%d q-blocks %d: whole units\n", l.first, l.second, n), 1;
  for (int n : {64, 80, 128})
    if (!smaller(32, 8, n) || !smaller(28, 4, n)) return std::printf("groups, q-blocks %d: whole units\n", n), 1;
  for (int n : {1, 40, 47, 1024})
    if (smaller(32, 32, n) || smaller(32, 8, n) || smaller(28, 4, n)) return std::printf("q-blocks %d: smaller units\n", n), 1;
  const int cases[][4] = {
      // H, Hkv, q-block begin, q-block end
      {32, 8, 0, 1024}, {32, 8, 128, 256}, {28, 4, 0, 512}, {24, 24, 0, 931}, {4, 4, 0, 1},   {7, 1, 0, 19},
      {64, 1, 0, 33},   {71, 1, 0, 40},    {128, 1, 0, 17}, {128, 2, 3, 30},  {130, 1, 0, 9}, {96, 3, 0, 25},
      {1, 1, 0, 300},   {6, 3, 5, 6},      {256, 1, 0, 5},  {40, 8, 0, 77},
  };
  int bad = 0;
  for (const auto& c : cases) {
    const int H = c[0], Hkv = c[1], b = c[2], e = c[3];
    const long grid = (long)xattn::grid_for(H, Hkv, e - b);
    std::vector<int> seen((size_t)H * (e - b), 0);
    long stray = 0;
    for (long id = 0; id < grid; ++id) {
      int head = -1, qb = -1;
      if (!xattn::map_workgroup((int)id, H, Hkv, b, e, &head, &qb)) continue;
      if (head < 0 || head >= H || qb < b || qb >= e) {
        ++stray;
        continue;
      }
      ++seen[(size_t)head * (e - b) + (qb - b)];
    }
    long missing = 0, twice = 0;
    for (int v : seen) {
      missing += v == 0;
      twice += v > 1;
    }
    // the 64 ids that reach one XCD one after the other must share their KV head
    long mixed = 0;
    for (long u = 0; u * 512 < grid; ++u)
      for (int x = 0; x < 8; ++x) {
        int kv = -1;
        for (int w = 0; w < 64; ++w) {
          int head, qb;
          if (!xattn::map_workgroup((int)(u * 512 + w * 8 + x), H, Hkv, b, e, &head, &qb)) continue;
          const int g = head / (H / Hkv);
          if (kv >= 0 && g != kv) ++mixed;
          kv = g;
        }
      }
    std::printf("H=%d Hkv=%d q-blocks [%d,%d): grid %ld missing %ld twice %ld stray %ld mixed-units %ld\n", H, Hkv, b, e,
                grid, missing, twice, stray, mixed);
    bad += (missing || twice || stray || mixed) ? 1 : 0;
  }
  return bad ? 1 : 0;
}
