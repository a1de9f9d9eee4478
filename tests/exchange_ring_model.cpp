// Host model of the exchange between the workgroups of the tridiagonalisation: every workgroup a
// state machine that runs the rules of exchange_ring.h, one word per step, in any interleaving.
// Prints "ok" when every interleaving tried ends with each word read in its own column.
//   exchange_ring_model <rows> <workgroups> <columns> <rule>
// rule 0: as shipped; 1: a workgroup also gathers the column that publishes its last row.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "exchange_ring.h"

using namespace dftbhip;

struct Group {
  int p, gathers, k = 0, phase = 0, row = 0;   // phase 0 publish, 1 gather, 2 empty, 3 left
};

struct Model {
  int m, P, kEnd;
  std::vector<std::vector<int>> ring;   // column of the word in a slot, -1: empty
  std::vector<Group> g;
  const char* wrong = nullptr;

  Model(int m_, int P_, int kEnd_, int rule)
      : m(m_), P(P_), kEnd(kEnd_), ring(kRingSlots, std::vector<int>(m_, -1)) {
    for (int p = 0; p < P; ++p) {
      Group x{p, 0};
      const int last = ring_last_row(p, P, m);
      x.gathers = ring_gathers(last, kEnd);
      if (rule == 1 && last < kEnd) x.gathers = last;
      g.push_back(x);
    }
  }
  // one word of workgroup x; false: it waits, or has left
  bool step(Group& x) {
    std::vector<int>& now = ring[x.k % kRingSlots];
    if (x.phase == 0) {
      for (int r = x.p; r < m; r += P)
        if (ring_published(r, x.k)) {
          if (now[r] >= 0) wrong = "a word is published over one that was not emptied";
          now[r] = x.k;
        }
      x.phase = x.k == x.gathers ? 3 : 1;
      x.row = x.k + 1;
      return true;
    }
    if (x.phase == 1) {
      if (now[x.row] < 0) return false;
      if (now[x.row] != x.k) wrong = "a word of another column is read";
      if (++x.row == m) x.phase = 2;
      return true;
    }
    if (x.phase == 2) {
      for (int r = x.p; r < m; r += P)
        if (ring_emptied(r, x.k)) ring[(x.k + kRingSlots - 1) % kRingSlots][r] = -1;
      x.phase = ++x.k == kEnd || x.k > x.gathers ? 3 : 0;
      return true;
    }
    return false;
  }
  bool finished() const {
    for (const Group& x : g)
      if (x.phase != 3) return false;
    return true;
  }
};

// `late` runs a step only when no other workgroup can: every other one is as far ahead of it as
// the rules let it be
static const char* one_late(int m, int P, int kEnd, int rule, int late) {
  Model M(m, P, kEnd, rule);
  while (!M.wrong && !M.finished()) {
    bool any = false;
    for (Group& x : M.g)
      while (x.p != late && !M.wrong && M.step(x)) any = true;
    if (!any && !M.wrong && !M.step(M.g[late])) return "the workgroups wait for each other";
  }
  return M.wrong;
}

static const char* random_order(int m, int P, int kEnd, int rule, unsigned seed) {
  Model M(m, P, kEnd, rule);
  std::mt19937 rng(seed);
  while (!M.wrong && !M.finished()) {
    bool any = false;
    for (int tries = 0; tries < 8 * P && !any; ++tries) {
      Group& x = M.g[rng() % P];
      for (int burst = 1 + rng() % (4 * m); burst > 0 && !M.wrong && M.step(x); --burst) any = true;
    }
    if (any) continue;
    for (Group& x : M.g) any = any || M.step(x);
    if (!any) return "the workgroups wait for each other";
  }
  return M.wrong;
}

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  const int m = std::atoi(argv[1]), P = std::atoi(argv[2]), kEnd = std::atoi(argv[3]),
            rule = std::atoi(argv[4]);
  for (int late = 0; late < P; ++late)
    if (const char* w = one_late(m, P, kEnd, rule, late)) {
      std::printf("workgroup %d late: %s\n", late, w);
      return 1;
    }
  for (unsigned seed = 0; seed < 20; ++seed)
    if (const char* w = random_order(m, P, kEnd, rule, seed)) {
      std::printf("order %u: %s\n", seed, w);
      return 1;
    }
  std::puts("ok");
  return 0;
}
