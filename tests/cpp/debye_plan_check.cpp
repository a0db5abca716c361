// CPU checks of the runs of the direct Debye sums through moments
// (csrc/xs_debye_plan.h), built with g++ by tests/test_debye_plan.py.
//
// 1. The runs of a row's segment pairs cover its tile pairs' items exactly once,
//    in order, also where a segment pair has 2^32 and more of them.
// 2. tile_pair visits every tile pair of small segments once, and at the ends and
//    the row boundaries of large ones gives the row and column that hold it.
// 3. The inputs of the GPU tests of the moments take the moments.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <tuple>
#include <vector>

#include "xs_debye_plan.h"

using namespace xs;
using namespace xs::debye;

static int failures = 0;
#define CHECK(cond, ...)                 \
  do {                                   \
    if (!(cond)) {                       \
      ++failures;                        \
      std::printf("FAIL: " __VA_ARGS__); \
      std::printf("\n");                 \
    }                                    \
  } while (0)

static uint64_t tiles(uint64_t n) { return (n + kMTile - 1) / kMTile; }

static void check_runs(const std::vector<uint32_t> &cnt, unsigned n_el, unsigned nblocks, int cus) {
  const RunTables T = plan_runs(cnt, n_el, nblocks, cus);
  uint64_t total = 0, expect = 0, next = 0;
  for (uint32_t a = 0; a < cnt.size(); ++a)
    for (uint32_t b = a; b < cnt.size(); ++b)
      expect += (a == b ? tiles(cnt[a]) * (tiles(cnt[a]) + 1) / 2 : tiles(cnt[a]) * tiles(cnt[b])) << T.shift;
  for (size_t i = 0; i < T.runs.size(); ++i) {
    const Run &r = T.runs[i];
    const bool same = i && T.runs[i - 1].offA == r.offA && T.runs[i - 1].offB == r.offB;
    const uint64_t all = (r.diag ? tiles(r.cntA) * (tiles(r.cntA) + 1) / 2 : tiles(r.cntA) * tiles(r.cntB)) << T.shift;
    CHECK(r.first == (same ? next : 0), "run %zu starts at %llu", i, (unsigned long long)r.first);
    CHECK(r.count > 0 && r.first + r.count <= all, "run %zu", i);
    next = r.first + r.count;
    const bool last = i + 1 == T.runs.size() || T.runs[i + 1].offA != r.offA || T.runs[i + 1].offB != r.offB;
    CHECK(!last || next == all, "segment pair ends at %llu of %llu", (unsigned long long)next,
          (unsigned long long)all);
    total += r.count;
  }
  CHECK(total == expect, "%llu items of %llu", (unsigned long long)total, (unsigned long long)expect);
  const size_t rows = (size_t)n_el * (n_el + 1) / 2 * nblocks * (nblocks + 1) / 2;
  CHECK(T.row_run.size() == rows + 1 && T.row_run[rows] == T.runs.size(), "rows");
  CHECK(T.runs.size() <= max_runs(rows, cus), "%zu runs", T.runs.size());
  for (size_t r = 0; r < rows; ++r) CHECK(T.row_run[r] <= T.row_run[r + 1], "row %zu", r);
  std::printf("runs of %zu segments: %zu, items %llu\n", cnt.size(), T.runs.size(),
              (unsigned long long)total);
}

// Inputs of the GPU tests of the moments (tests/test_gpu_debye_moments.py, _coherent.py):
// they must take them.  R: the diagonal of a box that the atoms nearly fill.
static void check_taken(const std::vector<uint32_t> &cnt, unsigned n_el, unsigned nblocks, double box,
                        double Q, unsigned nq) {
  for (double fill : {0.95, 1.0}) {
    MeshBox in;
    in.R = fill * box * std::sqrt(3.0);
    in.Q = Q;
    in.finite = true;
    MomentPlan plan;
    CHECK(plan_moments(in, cnt, n_el, nblocks, nq, 256, &plan), "pair by pair: box %g, q to %g", box, Q);
    CHECK(moments_lds_bytes(plan.bins.nb, plan.bins.K) <= kMLds, "LDS of %u bins", plan.bins.nb);
    std::printf("box %g q %g: %u bins, %d moments\n", box, Q, plan.bins.nb, plan.bins.K);
  }
}

int main() {
  check_taken({1500}, 1, 1, 30.0, 6.0, 400);
  check_taken({1, 1345, 63, 64, 65}, 5, 1, 40.0, 10.0, 1024);
  check_taken({1281, 700}, 2, 1, 25.0, 12.0, 777);
  check_taken({2000, 513}, 2, 1, 120.0, 25.0, 1000);
  check_taken({3000}, 1, 1, 300.0, 20.0, 1500);
  check_taken({1500, 321}, 2, 1, 35.0, 14.0, 300);
  check_taken({400, 400, 400, 300, 300, 300}, 2, 3, 35.0, 14.0, 300);
  check_taken({1000, 3000}, 2, 1, 10.03, 20.0, 300);
  check_taken({8192, 8192}, 2, 1, 10.03, 2.0, 300);
  check_runs({1}, 1, 1, 256);
  check_runs({64, 65, 0, 1}, 4, 1, 256);
  check_runs({700, 30, 5000, 64, 0, 129}, 2, 3, 256);
  check_runs({92681u * 64u}, 1, 1, 256);       // 2^32 - 2^14 ... tile pairs
  check_runs({92682u * 64u}, 1, 1, 256);       // 2^32 and more
  check_runs({65536u * 64u, 65537u * 64u}, 2, 1, 256);
  check_runs({6000000u, 100u, 7000001u}, 3, 1, 256);
  for (uint32_t TB : {1u, 2u, 3u, 17u, 100u}) {
    std::set<std::pair<uint32_t, uint32_t>> seen;
    for (uint64_t tp = 0; tp < (uint64_t)TB * (TB + 1) / 2; ++tp) {
      const TilePair p = tile_pair(tp, TB, true);
      CHECK(p.ti <= p.tj && p.tj < TB && seen.insert({p.ti, p.tj}).second, "pair %llu of %u",
            (unsigned long long)tp, TB);
    }
  }
  for (uint32_t TB : {92682u, 1000003u, 33554432u}) {
    std::mt19937_64 rng(TB);
    auto first = [&](uint64_t i) { return i * TB - i * (i - 1) / 2; };  // of row i
    for (int k = 0; k < 2000; ++k) {
      const uint64_t i = k < 3 ? (uint64_t)k : k < 6 ? TB - 1 - (k - 3) : rng() % TB;
      const TilePair a = tile_pair(first(i), TB, true), b = tile_pair(first(i) + (TB - 1 - i), TB, true);
      CHECK(a.ti == i && a.tj == i && b.ti == i && b.tj == TB - 1, "row %llu of %u", (unsigned long long)i, TB);
    }
    const TilePair c = tile_pair((uint64_t)TB * TB - 1, TB, false);
    CHECK(c.ti == TB - 1 && c.tj == TB - 1, "last of %u", TB);
  }
  if (failures) {
    std::printf("%d failures\n", failures);
    return 1;
  }
  std::printf("ok\n");
  return 0;
}
