// Host check of what the scan's threads read (scan_pair, mdmc_tilemap.h):
// workgroups of whole cell planes (any first segment) and of whole tiles, over
// random segment counts.  Every segment is read by its own thread, and nothing
// past the first padding entry is read at all.
#include "mdmc_tilemap.h"

#include <algorithm>
#include <cstdio>
#include <random>

int main() {
  constexpr uint32_t kTile = 2048, kIpt = 8;
  std::mt19937 rng(5);
  for (int it = 0; it < 3000; ++it) {
    const bool planes = it % 3 != 0;
    uint32_t per, n;  // segments per workgroup and in all
    if (planes) {
      const uint32_t plane = 1u + rng() % (it % 2 ? 2048u : 40u), cz = 1u + rng() % (it % 2 ? 40u : 1400u);
      per = kTile / plane * plane;
      n = plane * cz;
    } else {
      per = kTile;
      n = 1u + rng() % 200000u;
    }
    if (it == 1) { per = 2046u; n = 4095u; }
    for (uint32_t first = 0; first < n; first += per) {
      const uint32_t end = std::min(first + per, n);
      for (uint32_t t = 0; t < 256u; ++t) {
        const uint32_t base = first + t * kIpt;
        for (uint32_t i = 0; i < kIpt / 2u; ++i) {
          const uint32_t at = mdmc::scan_pair(base, i, end);
          if (at + 1u > n || (base + 2u * i < end && at != base + 2u * i)) {
            std::printf("n %u per %u first %u thread %u pair %u reads %u\n", n, per, first, t, i, at);
            return 1;
          }
        }
      }
    }
  }
  std::printf("OK\n");
  return 0;
}
