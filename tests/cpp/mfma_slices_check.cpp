// CPU checks of the int8 slices of the sinc values (csrc/xs_mfma_plan.h), built with
// g++ by tests/test_mfma_slices.py.
//
// Values that |q| r > kTopSliceX allows, |v| <= 1 / (kTopSliceX - 1e-8), have an empty top
// slice, to the last one and of either sign; some at 1/129 do not.
// The plan of a call of its own (wide: waves side by side, columns of fewer slices in the
// groups of more): every pair type one column of one group, slices that cover its count,
// a k range that covers its bins, slices that do not overlap.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "xs_mfma_plan.h"

using namespace xs;

static int failures = 0;
#define CHECK(cond, ...)                 \
  do {                                   \
    if (!(cond)) {                       \
      ++failures;                        \
      std::printf("FAIL: " __VA_ARGS__); \
      std::printf("\n");                 \
    }                                    \
  } while (0)

static long long top(double v) { return ((long long)std::rint(std::ldexp(v, 34)) + kSliceBias) >> 28; }

static void check_wide(unsigned ntypes, unsigned seed, int maxbits) {
  std::mt19937_64 rng(seed);
  std::vector<unsigned long long> off(ntypes), bound(ntypes);
  std::vector<uint32_t> nh(ntypes);
  for (unsigned t = 0; t < ntypes; ++t) {
    nh[t] = (uint32_t)(rng() % 5000);  // (an extent: 0 for empty columns)
    off[t] = 5000ull * t;
    const int bits = (int)(rng() % maxbits);
    bound[t] = nh[t] && bits ? (rng() & ((1ull << bits) - 1)) | (1ull << (bits - 1)) : 0;
  }
  MfmaBatchPlan p;
  CHECK(mfma_batch_plan(off, nh, bound, 300, &p, true), "refused (seed %u)", seed);
  std::vector<int> types(ntypes, 0), cols(ntypes, 0);
  for (const MfmaCol &c : p.cols) {
    ++types[c.type];
    CHECK(c.hist_off == off[c.type] && c.nhist == nh[c.type], "column of type %u", c.type);
  }
  unsigned long long b = 0;
  uint32_t tile = 0, launch = 0;
  for (const MfmaLaunch &L : p.launches) {
    CHECK(L.tile0 == tile && L.ntiles > 0 && L.nb >= 1 && L.nb <= (uint32_t)kMfmaMaxSlicesB &&
              (L.wn == 1 || L.wn == 2) && L.nt == (L.nb <= 2 ? 2u : 1u),
          "launch %u", launch);
    for (uint32_t g = L.tile0; g < L.tile0 + L.ntiles; ++g) {
      const MfmaTile &d = p.tiles[g];
      CHECK(d.b_off == b && d.ncol >= 1 && d.ncol <= 32 * L.nt * L.wn && d.kt >= 1, "group %u", g);
      b += (unsigned long long)L.nb * L.nt * L.wn * d.kt * 64;
      for (uint32_t c = d.col0; c < d.col0 + d.ncol; ++c) {
        ++cols[c];
        const MfmaCol &col = p.cols[c];
        CHECK((bound[col.type] >> (7 * L.nb)) == 0ull, "column %u: count", c);
        CHECK(32ull * d.kt >= col.nhist, "column %u: bins", c);
        CHECK(d.kt <= p.kt_max, "group %u: k range", g);
      }
    }
    tile += L.ntiles;
    ++launch;
  }
  CHECK(tile == p.tiles.size() && b * 16 == p.b_bytes && launch <= (uint32_t)kMfmaMaxSlicesB, "totals");
  for (unsigned t = 0; t < ntypes; ++t) CHECK(types[t] == 1 && cols[t] == 1, "type or column %u", t);
}

int main() {
  for (double x = kTopSliceX; x < 4 * kTopSliceX; x += 0.0137) {
    const double v = 1.0 / (x - 1e-8);
    CHECK(top(v) == 0 && top(-v) == 0 && top(0.3 * v) == 0, "value 1/%g", x);
  }
  CHECK(top(0.0) == 0, "0");
  CHECK(top(1.0 / 129.0) == 1 && top(1.0 / 129.02) == 0, "the bound");
  for (unsigned s = 0; s < 4000; ++s) check_wide(1 + s % 400, s, s % 3 ? 35 : 15);
  if (failures) {
    std::printf("%d failures\n", failures);
    return 1;
  }
  std::printf("ok\n");
  return 0;
}
