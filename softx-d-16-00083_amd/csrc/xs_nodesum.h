// Sine sums of many histograms over Chebyshev nodes (xs_nodesum.hip).
#pragma once

#include <cstddef>
#include <cstdint>

#include "xs_internal.h"

namespace xs {
namespace nodesum {

constexpr unsigned kNodes = 64;      // Chebyshev nodes of a group of bins
constexpr unsigned kMaxBins = 4096;  // bins of a group, at most
constexpr unsigned kRows = 16;       // histograms of a tile

// One histogram: its first bin, its bins and its row of S.
struct Row {
  unsigned long long hist_off;
  uint32_t nhist, srow;
};

// The groups of a call, found on the device from max |q|: bins per group, and
// whether the groups are compressed (else every bin is a node, 64 a group).
struct Plan {
  uint32_t bins, compress;
};

// Groups of a tile whose longest histogram has nhist bins, in groups of `bins`.
__host__ __device__ inline unsigned groups_for(unsigned nhist, unsigned bins) {
  return (nhist + bins - 1) / bins + 1;
}

__host__ __device__ inline unsigned align_groups(unsigned groups) { return (groups + 15u) & ~15u; }

// Up to this many histograms take few_kernel.
constexpr unsigned kFew = 8;

// Device memory of a call over tiles of 16 rows: the tables, then the weights of
// as many groups and tiles at a time as fit `budget` bytes (at least 16 groups).
struct Layout {
  size_t plan, rows, nmax, lagrange, node, weights, total;
  unsigned ntiles, nhist_max, group_cap;  // groups of the longest tile
  unsigned tiles_at_once, groups_at_once;
};
Layout layout(unsigned ntiles, unsigned nhist_max, size_t budget);

constexpr size_t kBudget = size_t(256) << 20;

// A call's memory (L.total bytes at mem) and its rows: ntypes histograms of
// nhist bins, whose tables are made here, or the caller's own (ntypes = 0):
// own_rows[16 ntiles], rows beyond the last with nhist 0 and nhist not rising
// from row to row, and own_nmax[ntiles], on the device.
struct Tables {
  Layout L;
  char *mem;
  unsigned ntypes, nhist;
  const Row *own_rows;
  const uint32_t *own_nmax;
  template <class T>
  T *at(size_t off) const {
    return reinterpret_cast<T *>(mem + off);
  }
  const Row *rows() const { return ntypes ? at<Row>(L.rows) : own_rows; }
  const uint32_t *nmax() const { return ntypes ? at<uint32_t>(L.nmax) : own_nmax; }
};

// S (nrows x nq) of the rows, overwritten.  Launches only (graph-capturable).
int run(xs_ctx *ctx, const Tables &T, const unsigned long long *hist, unsigned nrows, double bin,
        const double *q, unsigned nq, double *S);

}  // namespace nodesum

// S (nrows x nq) of rows (on the device) bin by bin, overwritten (xs_iq.hip); launches
// only, no memory of its own.  pairsum_short: where that is the faster form.
bool pairsum_short(const xs_ctx *ctx, size_t nrows, unsigned nhist_max, unsigned nq);
int pairsum_rows(xs_ctx *ctx, const unsigned long long *hist, const nodesum::Row *rows, unsigned nrows,
                 unsigned nhist_max, double bin, const double *q, unsigned nq, double *S);

}  // namespace xs
