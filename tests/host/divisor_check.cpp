// Host-only check of divisions by products (attn_tiles.h): exact for every number below 2^31.  Exit status 0 when all hold.
#include <cstdio>

#include "attn_tiles.h"

int main() {
  long wrong = 0, checked = 0;
  uint32_t seed = 1;
  for (uint32_t i = 1; i < 6000; ++i) {
    const uint32_t d = i < 5000 ? i : (0x7fffffffu - (i - 5000) * 7919u);
    const xattn::Divisor v = xattn::divisor(d);
    const uint32_t most = 0x7fffffffu / d;
    auto check = [&](uint32_t x) {
      wrong += xattn::divided(x, v) != x / d;
      ++checked;
    };
    for (uint32_t q : {0u, 1u, 2u, most / 2, most}) {
      if (q > most) continue;
      check(q * d);
      if (q) check(q * d - 1);
      if (q * (uint64_t)d + d - 1 <= 0x7fffffffu) check(q * d + d - 1);
    }
    check(0x7fffffffu);
    for (int k = 0; k < 50; ++k) check((seed = seed * 1664525u + 1013904223u) >> 1);
  }
  std::printf("%ld quotients, %ld wrong\n", checked, wrong);
  return wrong ? 1 : 0;
}
