// CPU checks of a batch plan's run buffer (csrc/xs_batch_layout.h), built with
// g++ by tests/test_batch_layout.py.  Over every pair of forms that two calls on
// one plan can have (host or device arrays, with or without pair sums and PDFs,
// pair sums over the nodes, on the matrix cores or without node tables, two nq):
// 1. the kept regions (rows, lengths, PDF descriptors, matrix-core tables) lie at
//    the same places in both;
// 2. nothing that one form writes overlaps what the other keeps;
// 3. the regions of one form are aligned to 256 bytes, disjoint and inside it.
#include <cstdio>
#include <utility>
#include <vector>

#include "xs_batch_layout.h"

using namespace xs;
typedef std::pair<size_t, size_t> Range;  // first byte, bytes

struct Form {
  RunLayout L;
  std::vector<Range> kept, written;
};

static Form form(bool host, bool S, bool pdf, int sums, size_t nq, size_t types) {
  RunSizes n;
  n.rows = (types + 15) / 16 * 16 * 16;
  n.nmax = (types + 15) / 16 * 4;
  n.pdfdesc = (types + 2) / 3 * 232;
  n.mm_cols = types * 16;
  n.mm_tiles = types * 24;
  if (host) {
    n.q = S ? nq * 8 : 0;
    n.hist = types * 1001 * 8;
    n.S = S ? types * nq * 8 : 0;
    n.pdf = pdf ? types * 1001 * 8 : 0;
  }
  if (S && sums == 1) {
    n.mm_a = 5 * 4096 * nq;
    n.mm_b = types * 2048;
  }
  if (S && sums == 0) n.nodes = 2100000 + types * 1024;
  const RunLayout L = run_layout(n);
  return Form{L,
              {{L.rows, n.rows}, {L.nmax, n.nmax}, {L.pdfdesc, n.pdfdesc}, {L.mm_cols, n.mm_cols},
               {L.mm_tiles, n.mm_tiles}},
              {{L.q, n.q}, {L.hist, n.hist}, {L.S, n.S}, {L.pdf, n.pdf}, {L.mm_a, n.mm_a},
               {L.mm_b, n.mm_b}, {L.nodes, n.nodes}}};
}

static bool overlap(const Range &a, const Range &b) {
  return a.second && b.second && a.first < b.first + b.second && b.first < a.first + a.second;
}

int main() {
  int failures = 0;
  for (size_t types : {size_t(1), size_t(3), size_t(16), size_t(17), size_t(48 * 6)}) {
    std::vector<Form> f;
    for (int bits = 0; bits < 8; ++bits)
      for (int sums = 0; sums < 3; ++sums)
        for (size_t nq : {size_t(1), size_t(600)}) f.push_back(form(bits & 1, bits & 2, bits & 4, sums, nq, types));
    for (size_t i = 0; i < f.size(); ++i) {
      std::vector<Range> all = f[i].kept;
      all.insert(all.end(), f[i].written.begin(), f[i].written.end());
      for (size_t a = 0; a < all.size(); ++a) {
        if (all[a].first % 256 || all[a].first + all[a].second > f[i].L.total) ++failures;
        for (size_t b = 0; b < a; ++b) failures += overlap(all[a], all[b]);
      }
      for (size_t j = 0; j < f.size(); ++j) {
        failures += f[i].kept != f[j].kept;
        for (const Range &w : f[i].written)
          for (const Range &k : f[j].kept) failures += overlap(w, k);
      }
    }
    std::printf("types=%zu forms=%zu\n", types, f.size());
  }
  if (failures) {
    std::printf("%d failures\n", failures);
    return 1;
  }
  std::printf("ok\n");
  return 0;
}
