// Layout of a batch plan's run buffer.  Plain C++ (no HIP), so that the same
// code builds into libxs_hip and into CPU tests of the layout.
//
// The buffer holds two kinds of regions.  Kept ones are uploaded when they
// change and read by every later run and graph replay: the pair types' rows,
// the PDF descriptors, the matrix-core tables.  The others are written by
// each run before it reads them.  The kept regions come first, at places that
// only the plan decides, so that no run of another form (host or device,
// with or without PDFs, on the matrix cores or over the nodes) writes there.
#pragma once

#include <cstddef>

namespace xs {

struct RunLayout {
  size_t rows, nmax, pdfdesc, mm_cols, mm_tiles;  // kept
  size_t q, hist, S, pdf, mm_a, mm_b, nodes;      // of a run
  size_t total;
};

// Bytes of the kept regions (of a plan) and of a run's own (0: not needed).
struct RunSizes {
  size_t rows = 0, nmax = 0, pdfdesc = 0, mm_cols = 0, mm_tiles = 0;
  size_t q = 0, hist = 0, S = 0, pdf = 0, mm_a = 0, mm_b = 0, nodes = 0;
};

inline RunLayout run_layout(const RunSizes &n) {
  RunLayout L{};
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off = (off + bytes + 255) / 256 * 256;
    return at;
  };
  L.rows = take(n.rows);
  L.nmax = take(n.nmax);
  L.pdfdesc = take(n.pdfdesc);
  L.mm_cols = take(n.mm_cols);
  L.mm_tiles = take(n.mm_tiles);
  L.q = take(n.q);
  L.hist = take(n.hist);
  L.S = take(n.S);
  L.pdf = take(n.pdf);
  L.mm_a = take(n.mm_a);
  L.mm_b = take(n.mm_b);
  L.nodes = take(n.nodes);
  L.total = off;
  return L;
}

}  // namespace xs
