// CPU checks of the equal-count partition of few atoms over many bins
// (csrc/xs_hist_plan.h), built with g++ by tests/test_equal_count.py.
//
// 1. The device orders the atoms with a counter table per column: there are fewer
//    than 2 columns an atom, however wide the structure (up to 2^31 bins).
// 2. The tiles are those of the partition by the window's width alone (slabs and
//    columns as wide as it allows), which leaves the columns beyond the atoms empty.
#include <cmath>
#include <cstdio>
#include <vector>

#include "xs_hist_plan.h"

using namespace xs::hist;

int main() {
  int failures = 0;
  const uint32_t atoms[] = {1, 2, 3, 10, 999, 1024, 1025, 2000, 5000, 300000};
  for (uint32_t ne : atoms)
    for (double nhist : {1e4, 1e5, 1e6, 1e7, 1e8, 2e9})
      for (int shape = 0; shape < 4; ++shape)
        for (bool paired : {false, true}) {
          const double bin = 0.01, edge = nhist * bin / std::sqrt(3.0);
          const double box[6] = {0, 0, 0, edge, shape == 1 ? 1.0 : edge, shape >= 2 ? 0.0 : edge};
          const double cap = (32768 - 8) * bin / (2.0 * std::sqrt(3.0));
          uint32_t gx, gy, nz;
          choose_equal_count(ne, box, cap, paired, gx, gy, nz);
          if (!gx || !gy || !nz || (uint64_t)gx * gy >= 2ull * ne + 1) {
            ++failures;
            std::printf("FAIL: %u atoms, %g bins: %u x %u columns\n", ne, nhist, gx, gy);
            continue;
          }
          const double w = 0.9 * cap;
          const uint64_t nx = (uint64_t)std::max(1.0, std::ceil(edge / w)),
                         ny = (uint64_t)std::max(1.0, std::ceil((box[4] - box[1]) / w));
          // where no column may be empty the window decides nothing; elsewhere compare,
          // while there are columns few enough to go through
          if (nx * ny <= ne || nx * ny > 10000000) continue;
          std::vector<Tile> a, b;
          equal_count_tiles(7, ne, gx, gy, nz, paired, a);
          equal_count_tiles(7, ne, (uint32_t)nx, (uint32_t)ny, nz, paired, b);
          bool same = a.size() == b.size();
          for (size_t i = 0; same && i < a.size(); ++i) same = a[i].off == b[i].off && a[i].cnt == b[i].cnt;
          if (!same) {
            ++failures;
            std::printf("FAIL: %u atoms, %g bins: other tiles\n", ne, nhist);
          }
        }
  if (failures) {
    std::printf("%d failures\n", failures);
    return 1;
  }
  std::printf("ok\n");
  return 0;
}
