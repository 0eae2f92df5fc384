// Host check of how a wave's lanes hand each other values through LDS
// (mdmc_wave.h).  64 lanes run as coroutines, each alone as far as the next
// order point, in a fresh random sequence between two points: the loosest
// order the points allow.  Emit: sums in columns of the part, then vertices
// staged in the same words, then quads, twice over as for two chunks.
// Classify: a list filled by all lanes and taken a cell per lane, with row
// words beside it.  Everything must come out as with lanes in step.
#include "mdmc_wave.h"

#include <ucontext.h>

#include <algorithm>
#include <cstdio>
#include <functional>
#include <random>
#include <vector>

namespace {

constexpr uint32_t kLanes = 64, kRing = 512;

struct Wave {
  std::vector<ucontext_t> ctx = std::vector<ucontext_t>(kLanes);
  std::vector<std::vector<char>> stack = std::vector<std::vector<char>>(kLanes, std::vector<char>(65536));
  std::vector<bool> done = std::vector<bool>(kLanes, false);
  ucontext_t main;
  uint32_t cur = 0;
  std::function<void(uint32_t)> body;
};
Wave *g_wave = nullptr;

void lane_main() {
  g_wave->body(g_wave->cur);
  g_wave->done[g_wave->cur] = true;
  swapcontext(&g_wave->ctx[g_wave->cur], &g_wave->main);
}

struct Order {
  void operator()() const { swapcontext(&g_wave->ctx[g_wave->cur], &g_wave->main); }
};

void run(std::function<void(uint32_t)> body, std::mt19937 &rng) {
  Wave w;
  w.body = std::move(body);
  g_wave = &w;
  for (uint32_t l = 0; l < kLanes; ++l) {
    getcontext(&w.ctx[l]);
    w.ctx[l].uc_stack.ss_sp = w.stack[l].data();
    w.ctx[l].uc_stack.ss_size = w.stack[l].size();
    w.ctx[l].uc_link = nullptr;
    makecontext(&w.ctx[l], lane_main, 0);
  }
  std::vector<uint32_t> seq(kLanes);
  for (uint32_t l = 0; l < kLanes; ++l) seq[l] = l;
  for (bool any = true; any;) {
    any = false;
    std::shuffle(seq.begin(), seq.end(), rng);
    for (uint32_t l : seq) {
      if (w.done[l]) continue;
      w.cur = l;
      swapcontext(&w.main, &w.ctx[l]);
      any = true;
    }
  }
}

bool emit(std::mt19937 &rng) {
  uint32_t part[768] = {};
  std::vector<uint32_t> nv(kLanes), dv(kLanes), nq(kLanes), dq(kLanes), verts[2], quads[2];
  uint32_t V = 0, Q = 0;
  for (uint32_t l = 0; l < kLanes; ++l) {
    nv[l] = 1u + rng() % 4u;
    nq[l] = rng() % 4u;
    dv[l] = V;
    dq[l] = Q;
    V += nv[l];
    Q += nq[l];
  }
  for (auto &v : verts) v.assign(3 * V, 0u);
  for (auto &q : quads) q.assign(4 * Q, 0u);
  auto vword = [](uint32_t c, uint32_t l, uint32_t i, uint32_t k) { return 1u + k + 3u * i + 16u * l + 4096u * c; };
  auto qword = [](uint32_t c, uint32_t l, uint32_t i, uint32_t k) { return 1u + k + 4u * i + 16u * l + 4096u * c + (1u << 20); };
  auto copy = [&](std::vector<uint32_t> &out, uint32_t l) {  // four words a lane, then single ones
    const uint32_t words = (uint32_t)out.size(), tail = words & ~3u;
    for (uint32_t i = 4 * l; i < tail; i += 4 * kLanes) std::copy(part + i, part + i + 4, out.begin() + i);
    for (uint32_t i = tail + l; i < words; i += kLanes) out[i] = part[i];
  };
  run([&](uint32_t l) {
    for (uint32_t c = 0; c < 2; ++c) {
      for (uint32_t k = 0; k < 3; ++k) part[k * kLanes + l] = vword(c, l, 0, k);  // the lane's sums
      const uint32_t r[3] = {part[l], part[kLanes + l], part[2 * kLanes + l]};
      mdmc::wave_exchange(
          [&] {
            for (uint32_t i = 0; i < nv[l]; ++i)
              for (uint32_t k = 0; k < 3; ++k) part[3 * (dv[l] + i) + k] = i ? vword(c, l, i, k) : r[k];
          },
          [&] { copy(verts[c], l); }, Order());
      mdmc::wave_exchange(
          [&] {
            for (uint32_t i = 0; i < nq[l]; ++i)
              for (uint32_t k = 0; k < 4; ++k) part[4 * (dq[l] + i) + k] = qword(c, l, i, k);
          },
          [&] { copy(quads[c], l); }, Order());
    }
  }, rng);
  for (uint32_t c = 0; c < 2; ++c)
    for (uint32_t l = 0; l < kLanes; ++l) {
      for (uint32_t i = 0; i < 3 * nv[l]; ++i)
        if (verts[c][3 * dv[l] + i] != vword(c, l, i / 3, i % 3)) return false;
      for (uint32_t i = 0; i < 4 * nq[l]; ++i)
        if (quads[c][4 * dq[l] + i] != qword(c, l, i / 4, i % 4)) return false;
    }
  return true;
}

bool classify(std::mt19937 &rng) {
  constexpr uint32_t kRows = 24;
  uint16_t ring[kRing] = {};
  uint32_t row_word[kRows] = {}, act[kRows][kLanes], first[kRows][kLanes], have[kRows + 1] = {0};
  std::vector<uint32_t> want, got;
  for (uint32_t m = 0; m < kRows; ++m) {
    have[m + 1] = have[m];
    for (uint32_t l = 0; l < kLanes; ++l) {
      act[m][l] = m % 5u == 0u ? 15u : rng() & rng() & 15u;
      first[m][l] = have[m + 1];
      for (uint32_t q = 0; q < 4; ++q)
        if ((act[m][l] >> q) & 1u) {
          want.push_back((m << 10 | (4u * l + q)) + (m + 1u) * 65536u);
          ++have[m + 1];
        }
    }
  }
  got.assign(want.size(), 0u);
  run([&](uint32_t l) {
    uint32_t done = 0;
    auto drain = [&](uint32_t n) {
      const uint32_t e = mdmc::ring_take<kRing>(ring, done, l, n, Order());
      if (l < n) got[done + l] = e + row_word[e >> 10] * 65536u;
      done += n;
    };
    for (uint32_t m = 0; m < kRows; ++m) {
      if (l == 0) row_word[m] = m + 1u;
      uint32_t pos = first[m][l];
      for (uint32_t q = 0; q < 4; ++q)
        if ((act[m][l] >> q) & 1u) ring[pos++ % kRing] = (uint16_t)(m << 10 | (4u * l + q));
      while (have[m + 1] - done >= kLanes) drain(kLanes);
    }
    if (have[kRows] != done) drain(have[kRows] - done);
  }, rng);
  return got == want;
}

}  // namespace

int main() {
  std::mt19937 rng(7);
  for (int it = 0; it < 100; ++it) {
    if (!emit(rng)) { std::printf("emit %d\n", it); return 1; }
    if (!classify(rng)) { std::printf("classify %d\n", it); return 1; }
  }
  std::printf("OK\n");
  return 0;
}
