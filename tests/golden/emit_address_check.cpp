// Host check of the emit's address arithmetic (mdmc_tilemap.h): division by
// multiplication against the division, and that every byte offset a lane forms
// for a segment within emit_span of its wave's first one fits in 32 bits.
#include "mdmc_tilemap.h"

#include <cstdio>
#include <random>

int main() {
  std::mt19937_64 rng(3);
  for (int it = 0; it < 200000; ++it) {
    uint32_t d = it < 70000 ? (uint32_t)it + 1u : (uint32_t)(rng() >> (32 + it % 32));
    if (d == 0) d = 1;
    const mdmc::FastDiv f = mdmc::fast_div(d);
    const uint32_t top = 0xFFFFFFFFu / d * d;  // the largest multiple
    const uint32_t ns[] = {0u, 1u, d - 1u, d, d + 1u, top - 1u, top, 0xFFFFFFFEu, 0xFFFFFFFFu, (uint32_t)rng(), (uint32_t)rng()};
    for (uint32_t n : ns)
      if (mdmc::div_by(n, f) != n / d) { std::printf("%u / %u\n", n, d); return 1; }
  }
  const uint32_t caps[] = {64u, 128u, 256u, 512u, 1024u};
  for (int it = 0; it < 200000; ++it) {
    const uint32_t cap = caps[rng() % 5];
    const uint64_t X = 2u + rng() % (1ull << (1 + rng() % 31)), cy = 1u + rng() % (1ull << (rng() % 24));
    if (X * (cy + 1u) > 0xFFFFFFFFull) continue;
    const uint64_t XT = (X - 1u + cap - 1u) / cap, Y = cy + 1u;
    const uint64_t span = mdmc::emit_span((uint32_t)X, (uint32_t)XT, cap);
    for (int r = 0; r < 4; ++r) {
      const uint64_t d = r == 0 ? span : r == 1 ? 0 : rng() % (span + 1), s0 = rng() % (XT * cy * 2);
      const uint64_t row0 = s0 / XT, xt0 = s0 % XT, row = (s0 + d) / XT, xt = (s0 + d) % XT;
      const uint64_t prow = (row / cy - row0 / cy) * Y + row % cy - row0 % cy;
      const uint64_t last = xt * cap + cap < X ? xt * cap + cap : X;  // past the tile's cells
      const uint64_t field = (prow * X + last - xt0 * cap) * 4u, rec = (d * cap + cap) * 4u;
      if (field + 8u > 0xFFFFFFFFull || rec + 8u > 0xFFFFFFFFull) {
        std::printf("X %llu cy %llu cap %u d %llu\n", (unsigned long long)X, (unsigned long long)cy, cap, (unsigned long long)d);
        return 1;
      }
    }
  }
  std::printf("OK\n");
  return 0;
}
