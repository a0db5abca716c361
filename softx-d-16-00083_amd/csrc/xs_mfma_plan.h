// Host-side planning of the batched matrix-core pair sums (xs_batch_run with
// XS_PAIRSUM_MFMA): the column order, the column groups and their slice
// layout.  Plain C++ (no HIP), so that the same code builds into libxs_hip
// and into CPU tests of the tables.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace xs {

constexpr int kMfmaSlicesA = 5;      // int8 slices of the sinc matrix
constexpr int kMfmaMaxSlicesB = 5;   // 7-bit count slices (counts below 2^35)

// A sinc value v is sliced as N + kSliceBias, N = rint(2^34 v): four 7-bit fields (less
// 64) and the bits from 28 on as the top slice.  That one is 0 for -127.0 < 1/v or
// 1/v > 129.016 (N + bias from 0 to 2^28), so beyond |q| r = kTopSliceX whatever the sine.
constexpr long long kSliceBias = 64ll * (1 + 128 + 16384 + 2097152);
constexpr double kTopSliceX = 130.0;

// Columns are the pair types, sorted by count slices (most first) and then
// by bin count (largest first), so that every group of NT column tiles of 32
// columns shares one slice count and one k range (its largest bin count).
struct MfmaCol {
  unsigned long long hist_off;  // first bin of the column's histogram
  uint32_t nhist, type;         // its bin count; its row of S
};
struct MfmaTile {
  unsigned long long b_off;  // first count slice of the group, in 16-byte units
  uint32_t kt, col0, ncol;   // k tiles of 32 bins; first column (sorted order); columns
  uint32_t pad;
};
struct MfmaLaunch {
  uint32_t tile0, ntiles, nb, nt;  // groups [tile0, tile0 + ntiles), slices, tiles a wave
  uint32_t wn;                     // waves side by side: a group has 32 nt wn columns
};
struct MfmaBatchPlan {
  std::vector<MfmaCol> cols;
  std::vector<MfmaTile> tiles;
  std::vector<MfmaLaunch> launches;
  uint32_t kt_max = 0;  // k tiles of the sinc slices (largest bin count)
  uint32_t nq = 0;
  size_t a_bytes = 0, b_bytes = 0;
};

// Builds the plan from each pair type's histogram offset, bin count and an
// upper bound of its counts (its pair count).  False if a bound reaches 2^35
// (more count slices than the kernels take).  A group holds 32 NT columns of
// one slice count (NT = 2 for up to two slices, else 1: more accumulators
// would not fit), never columns of the next.  Its slices are laid out
// [nb][NT][kt][64] (16-byte units) at b_off; the sinc slices take
// kMfmaSlicesA x MT x kt_max KiB, MT = 4 ceil(nq / 128).
// wide: a group may be two waves' tiles side by side (where there are columns for
// both), and columns of fewer slices join those of more while together they fit one
// such group, which saves a pass over the sinc slices.
inline bool mfma_batch_plan(const std::vector<unsigned long long> &hist_off,
                            const std::vector<uint32_t> &nhist,
                            const std::vector<unsigned long long> &count_bound, unsigned nq,
                            MfmaBatchPlan *plan, bool wide = false) {
  MfmaBatchPlan p;
  const size_t n = nhist.size();
  std::vector<uint32_t> nb(n);
  for (size_t t = 0; t < n; ++t) {
    uint32_t k = 1;
    while (k < (uint32_t)kMfmaMaxSlicesB && (count_bound[t] >> (7 * k)) != 0ull) ++k;
    if ((count_bound[t] >> (7 * k)) != 0ull) return false;
    nb[t] = k;
  }
  std::vector<uint32_t> order(n);
  for (size_t t = 0; t < n; ++t) order[t] = (uint32_t)t;
  std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) {
    return nb[a] != nb[b] ? nb[a] > nb[b] : nhist[a] > nhist[b];
  });
  struct Class {
    size_t c0, c1;
    uint32_t nb;
  };
  std::vector<Class> classes;
  for (size_t c = 0; c < n; ++c) {
    const uint32_t k = nb[order[c]];
    if (classes.empty() || classes.back().nb != k) {
      if (wide && !classes.empty() && c - classes.back().c0 < 64 * (classes.back().nb <= 2 ? 2u : 1u)) {
        size_t e = c;
        while (e < n && nb[order[e]] == k) ++e;
        if (e - classes.back().c0 <= 64 * (classes.back().nb <= 2 ? 2u : 1u)) {
          classes.back().c1 = e;
          std::stable_sort(order.begin() + classes.back().c0, order.begin() + e,
                           [&](uint32_t a, uint32_t b) { return nhist[a] > nhist[b]; });
          c = e - 1;
          continue;
        }
      }
      classes.push_back(Class{c, c, k});
    }
    classes.back().c1 = c + 1;
  }
  p.cols.resize(n);
  for (size_t c = 0; c < n; ++c) p.cols[c] = MfmaCol{hist_off[order[c]], nhist[order[c]], order[c]};
  unsigned long long b_off = 0;
  uint32_t max_nh = 0;
  for (const Class &cl : classes) {
    const uint32_t NT = cl.nb <= 2 ? 2 : 1;
    const uint32_t WN = wide && cl.c1 - cl.c0 > 32 * NT ? 2 : 1;
    MfmaLaunch L{(uint32_t)p.tiles.size(), 0u, cl.nb, NT, WN};
    for (size_t g = cl.c0; g < cl.c1; g += 32 * NT * WN) {
      const uint32_t kt = std::max<uint32_t>(1u, (nhist[order[g]] + 31) / 32);
      const uint32_t ncol = (uint32_t)std::min<size_t>(32 * NT * WN, cl.c1 - g);
      p.tiles.push_back(MfmaTile{b_off, kt, (uint32_t)g, ncol, 0u});
      b_off += (unsigned long long)cl.nb * NT * WN * kt * 64;
      max_nh = std::max(max_nh, nhist[order[g]]);
      ++L.ntiles;
    }
    p.launches.push_back(L);
  }
  const unsigned MT = (nq + 127) / 128 * 4;
  p.kt_max = std::max<uint32_t>(1u, (max_nh + 31) / 32);
  p.nq = nq;
  p.a_bytes = (size_t)kMfmaSlicesA * MT * p.kt_max * 1024;
  p.b_bytes = (size_t)b_off * 16;
  *plan = std::move(p);
  return true;
}

}  // namespace xs
