// Direct Debye sums through Chebyshev moments (xs_debye_moments.hip).
#pragma once

#include <vector>

#include "xs_internal.h"
#include "xs_nodes.h"

namespace xs {
namespace debye {

constexpr int kMaxMoments = 24;

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

// Whether the moments take fewer cycles than debye_kernel for these inputs
// (and fit), and with how many of them.  seg_cnt: atoms of each (element,
// block), element-major.
bool plan_moments(const MeshBox &in, const std::vector<uint32_t> &seg_cnt, unsigned n_el,
                  unsigned nblocks, unsigned nq, int cus, MomentPlan *plan);

// Bytes of the run tables, an upper bound.
size_t moments_table_bytes(const std::vector<uint32_t> &seg_cnt, unsigned n_el, unsigned nblocks,
                           int cus);

// Enqueues the call (all pointers device memory; S is overwritten).  `work`
// holds moments_table_bytes.  The pinned staging must be free.
int run_moments(xs_ctx *ctx, const MomentPlan &plan, const double *xyz, size_t n,
                const std::vector<uint32_t> &seg_cnt, unsigned n_el, unsigned nblocks,
                const MeshBox &in, const double *q, unsigned nq, double *S, void *work);

}  // namespace debye
}  // namespace xs
