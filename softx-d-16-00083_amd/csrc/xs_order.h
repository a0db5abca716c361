// Atoms into equal-count tiles on the device (xs_order.hip).
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

#include "xs_internal.h"

namespace xs {
namespace order {

// One element of a structure: atoms [start, start + n), its slabs along x and their
// share of the counters.
struct Seg {
  uint32_t start, n;
  uint32_t gx, slab0;      // slabs slab0 .. slab0 + gx - 1
  uint32_t count0, nb;     // buckets along x
  double lo[3], scale[3];  // 1 / extent (0 if flat)
};
// One slab: positions [start, start + n), its columns along y.
struct Slab {
  uint32_t start, n;
  uint32_t gy, col0;    // columns col0 .. col0 + gy - 1
  uint32_t seg;
  uint32_t count0, nb;  // buckets along y
  uint32_t zcount0, znb;  // buckets along z, of every column
};

// The tables of a set of elements, as the equal-count partition (gx slabs, gy columns
// in each) splits them.
struct Tables {
  std::vector<Seg> segs;
  std::vector<Slab> slabs;
  uint32_t ncols = 0;
  size_t natoms = 0, counters = 0;
  void add(uint32_t start, uint32_t n, uint32_t gx, uint32_t gy, const double box[6]);
  size_t table_bytes() const { return align_up(segs.size() * sizeof(Seg), 256) + slabs.size() * sizeof(Slab); }
  void write_tables(char *dst) const;  // table_bytes()
  size_t scratch_bytes() const;
};

// x, y, z in the final order (elements as they were, columns of a slab, atoms of a
// column along z) to sx, sy, sz.  tables: write_tables' bytes on the device.
template <class S, class T>
int run(xs_ctx *ctx, const Tables &t, const char *tables, char *scratch, const S *x, const S *y,
        const S *z, T *sx, T *sy, T *sz);

}  // namespace order
}  // namespace xs
