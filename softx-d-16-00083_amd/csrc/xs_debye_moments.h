// Direct Debye sums through Chebyshev moments (xs_debye_moments.hip).
#pragma once

#include <vector>

#include "xs_debye_plan.h"
#include "xs_internal.h"

namespace xs {
namespace debye {

// Enqueues the call (all pointers device memory; S is overwritten).  `work`
// holds moments_table_bytes.  The pinned staging must be free.
int run_moments(xs_ctx *ctx, const MomentPlan &plan, const double *xyz, size_t n,
                const std::vector<uint32_t> &seg_cnt, unsigned n_el, unsigned nblocks,
                const MeshBox &in, const double *q, unsigned nq, double *S, void *work);

}  // namespace debye
}  // namespace xs
