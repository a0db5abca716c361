// Host-side planning of the direct Debye sums through Chebyshev moments
// (xs_debye_moments.hip): whether to take them and with how many moments, and
// the runs of tile pairs that the work groups get.  Plain C++ (no HIP), so that
// the same code builds into libxs_hip and into CPU tests of the tables.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "xs_nodes.h"

namespace xs {
namespace debye {

constexpr int kMTile = 64;          // atoms per tile: one per lane
constexpr size_t kMLds = 160000;    // of the CU's 163,840 bytes
constexpr int kMaxMoments = 32;
constexpr int kMoments[] = {8, 10, 12, 14, 18, 24, 32};

// What the host knows of the inputs: the bounding-box diagonal R, max |q|,
// the mesh step and whether the mesh is uniform, and whether all coordinates
// and q are finite.
struct MeshBox {
  double R = 0, Q = 0, dq = 0;
  bool uniform = false, finite = false;
};

struct MomentPlan {
  nodes::Bins bins;
};

// A run of tile pairs of segments A and B: items first .. first + count,
// an item being a tile pair's share of jr J atoms.  64-bit: an element of
// 5.94 M atoms has 2^32 tile pairs.
struct Run {
  uint64_t first, count;
  uint32_t offA, cntA, offB, cntB, diag, pad;
};

struct RunTables {
  std::vector<Run> runs;
  std::vector<uint32_t> row_run;  // row r has the runs row_run[r] .. row_run[r + 1] - 1
  unsigned shift = 0;             // a tile pair is 2^shift items
};

inline size_t moments_lds_bytes(unsigned nb, int K) {
  return (size_t)nb * (K - 1) * 8 + ((size_t)nb * 4 + 7) / 8 * 8 + (size_t)K * 8;
}

// Cycles of the CUs for one call, to choose K and to leave small inputs to
// debye_kernel.  Measured: 199 cycles a wave of 64 pairs for K = 10 on the
// 8,000-atom rock-salt cube, the launch's start and end included, about 20 a
// moment (172 for K = 12 on 50,000 atoms, 14 a moment); the evaluation's sines
// at half the issue rate; 25 us for the launches and the copy of the tables.
inline double moments_cycles(double pairs, double rows, double rgroups, unsigned nq,
                             const nodes::Bins &b, double cus) {
  const double per_pair = 20.0 * b.K / 64.0;
  const double node_q = (double)b.entries() * nq * 2.0 * (27.0 * rgroups + 3.5 * rows) / 64.0;
  return pairs * per_pair / cus + node_q / cus + (double)b.entries() * 1.5 + 60000.0;
}
// 3.28 VALU instructions per pair and q at 67% issue, for q in blocks of 1,024
// whether filled or not (340 atoms, 714 q: 85 us; 594 atoms, 1,037 q: 107 us,
// against 50 us through the moments)
inline double direct_cycles(double pairs, unsigned nq, double cus) {
  return pairs * std::ceil(nq / 1024.0) * 1024.0 * (3.28 / 0.67) / 64.0 / cus + 60000.0;
}

// The runs of a call at most, and the bytes of their tables.
inline size_t max_runs(size_t rows, int cus) { return std::max<size_t>((unsigned)cus, 4 * rows); }
inline size_t moments_table_bytes(size_t rows, int cus) {
  return (max_runs(rows, cus) * sizeof(Run) + 255) / 256 * 256 + (rows + 1) * 4;
}

// Whether the moments take fewer cycles than debye_kernel for these inputs
// (and fit), and with how many of them.  seg_cnt: atoms of each (element,
// block), element-major.
inline bool plan_moments(const MeshBox &in, const std::vector<uint32_t> &seg_cnt, unsigned n_el,
                         unsigned nblocks, unsigned nq, int cus, MomentPlan *plan) {
  if (!in.finite || !(in.R > 1e-100 && in.R < 1e100) || !(in.Q > 1e-100 && in.Q < 1e100))
    return false;
  const unsigned nparts = nblocks * (nblocks + 1) / 2;
  const double rows = (double)(n_el * (n_el + 1) / 2) * nparts;
  double n = 0.0;
  for (uint32_t c : seg_cnt) n += c;
  const double pairs = 0.5 * n * (n - 1.0);
  const double rgroups = std::ceil(rows / 8.0);
  // a chunk of nodes per work group in x, rows in z, q blocks in y
  if (rows > 60000.0 || nq > 256u * 65535u) return false;
  double best = direct_cycles(pairs, nq, cus);
  bool found = false;
  for (int K : kMoments) {
    const nodes::Bins b = nodes::bins_for(in.R, in.Q, K);
    if (b.nb > 1000000u || moments_lds_bytes(b.nb, K) > kMLds) continue;
    // (a slab per run, and the rows' sums)
    const double slabs = ((double)max_runs((size_t)rows, cus) + rows) * (double)b.entries() * 8.0;
    if (slabs > (double)(size_t(1) << 30)) continue;
    const double c = moments_cycles(pairs, rows, rgroups, nq, b, cus);
    if (c < best) {
      best = c;
      plan->bins = b;
      found = true;
    }
  }
  return found;
}

// The runs of a call, by row (pair type, block pair).
inline RunTables plan_runs(const std::vector<uint32_t> &seg_cnt, unsigned n_el, unsigned nblocks,
                           int cus) {
  struct SegPair {
    uint32_t row, a, b;
  };
  RunTables T;
  const unsigned nparts = nblocks * (nblocks + 1) / 2;
  const unsigned nrows = n_el * (n_el + 1) / 2 * nparts;
  std::vector<uint32_t> off(seg_cnt.size() + 1, 0);
  for (size_t s = 0; s < seg_cnt.size(); ++s) off[s + 1] = off[s] + seg_cnt[s];
  // segment pairs by row: (element a, block i) with (element b, block j)
  std::vector<SegPair> sp;
  uint64_t total = 0;
  auto tiles = [&](uint32_t s) { return ((uint64_t)seg_cnt[s] + kMTile - 1) / kMTile; };
  auto pair_tiles = [&](const SegPair &v) {
    return v.a == v.b ? tiles(v.a) * (tiles(v.a) + 1) / 2 : tiles(v.a) * tiles(v.b);
  };
  unsigned p = 0;
  for (unsigned a = 0; a < n_el; ++a)
    for (unsigned c = a; c < n_el; ++c, ++p)
      for (unsigned i = 0; i < nblocks; ++i)
        for (unsigned j = i; j < nblocks; ++j) {
          const uint32_t row = p * nparts + nblocks * i - (i * (i + 1)) / 2 + j;
          const uint32_t ai = a * nblocks + i, cj = c * nblocks + j;
          sp.push_back(SegPair{row, ai, cj});
          if (a != c && i != j) sp.push_back(SegPair{row, a * nblocks + j, c * nblocks + i});
        }
  for (const SegPair &v : sp) total += pair_tiles(v);
  // shares of a tile pair, so that every wave of the chip has a few items
  while (T.shift < 3 && (total << T.shift) < 64ull * (unsigned)cus) ++T.shift;
  // runs: the shortest longest run for which the segment pairs' runs fill one
  // round of work groups (two runs a segment pair where those are many)
  const uint64_t most = std::max<uint64_t>((unsigned)cus, 2 * sp.size());
  double low = 0.0, per = std::max(1.0, (double)total);
  for (int it = 0; it < 50; ++it) {
    const double mid = 0.5 * (low + per);
    uint64_t nr = 0;
    for (const SegPair &v : sp) nr += (uint64_t)std::ceil((double)pair_tiles(v) / mid);
    (nr <= most ? per : low) = mid;
  }
  T.row_run.assign(nrows + 1, 0);
  for (const SegPair &v : sp) {
    const uint64_t t = pair_tiles(v) << T.shift;
    if (t) {
      const uint64_t nr = (uint64_t)std::ceil((double)pair_tiles(v) / per);
      uint64_t f = 0;
      for (uint64_t k = 0; k < nr; ++k) {
        const uint64_t e = t / nr * (k + 1) + t % nr * (k + 1) / nr;  // t (k + 1) / nr
        if (e == f) continue;
        T.runs.push_back(Run{f, e - f, off[v.a], seg_cnt[v.a], off[v.b], seg_cnt[v.b],
                             v.a == v.b ? 1u : 0u, 0u});
        f = e;
      }
    }
    T.row_run[v.row + 1] = (uint32_t)T.runs.size();
  }
  for (unsigned r = 0; r < nrows; ++r) T.row_run[r + 1] = std::max(T.row_run[r + 1], T.row_run[r]);
  return T;
}

// Tiles (ti, tj) of tile pair tp: of a segment with itself (diag), row ti holds
// the J tiles ti .. TB - 1, rows before it c(ti) pairs; else row ti all TB.
struct TilePair {
  uint32_t ti, tj;
};
#if defined(__HIPCC__)
__host__ __device__
#endif
inline TilePair tile_pair(uint64_t tp, uint32_t TB, bool diag) {
  if (!diag) return TilePair{(uint32_t)(tp / TB), (uint32_t)(tp % TB)};
  const double T2 = 2.0 * (double)TB + 1.0, d = T2 * T2 - 8.0 * (double)tp;
  const double g = floor(0.5 * (T2 - sqrt(d > 0.0 ? d : 0.0)));
  uint64_t i = g < 0.0 ? 0 : (uint64_t)g;
  if (i >= TB) i = TB - 1;
  auto c = [TB](uint64_t v) { return v * TB - v * (v - 1) / 2; };
  while (i > 0 && c(i) > tp) --i;
  while (i + 1 < TB && c(i + 1) <= tp) ++i;
  return TilePair{(uint32_t)i, (uint32_t)(i + (tp - c(i)))};
}

}  // namespace debye
}  // namespace xs
