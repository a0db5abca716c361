// Sine sums over Chebyshev nodes: host-side planning and the evaluation.
//
// A sum S(q) = sum_p f_q(r_p) over distances r_p in [0, R] with
// f_q(r) = (sin(q r)/q) (1/r - (e/q_c)/r^2), |q| <= Q, needs f_q only where
// it is known to FP64 accuracy between a few points: [0, R] is cut into nb
// bins of width h, and on a bin f_q is a Chebyshev series whose k-th
// coefficient is below 2 (Q h/4)^k / k! of its size (sin(q r)/(q r) is entire
// of exponential type q).  So the distances enter only through their
// Chebyshev moments T_0..T_{K-1} in each bin, whatever the number of q, and
// S(q) is the sum over the bins' K Chebyshev nodes of the moments turned into
// node weights times f_q(node).
#pragma once

#include <cmath>
#include <cstddef>
#include <cstdint>

namespace xs {
namespace nodes {

// Truncation: 2 (Q h/4)^K / K! at most this, per distance and relative to
// 1/(q r): an eighth of what rounding q r leaves of the farthest pair's sine, Q R 2^-53,
// or FP64 rounding.  (5e-13 was ten times what FP64 sums pair by pair leave.)
inline double truncation(double R, double Q) { return std::fmax(0x1p-52, Q * R * 0x1p-56); }

// The largest Q h/4 for K moments.
inline double reach(int K, double tol) {
  double f = 0.5 * tol;
  for (int k = 2; k <= K; ++k) f *= k;
  return std::pow(f, 1.0 / K);
}

// Bins of [0, R] for |q| <= Q with K moments: a distance is in units of the bins
// r inv_h, rounded once, and h = 1 / inv_h to 2^-64.
struct Bins {
  int K = 0;
  unsigned nb = 0;
  double inv_h = 0;
  long double h() const { return 1.0L / (long double)inv_h; }
  size_t entries() const { return ((size_t)nb + 1) * K; }  // one bin more: near pairs
};

inline Bins bins_for(double R, double Q, int K) {
  Bins b;
  b.K = K;
  b.inv_h = Q / (4.0 * reach(K, truncation(R, Q)));
  const double n = std::floor(R * b.inv_h * (1.0 + 1e-12)) + 1.0;
  b.nb = n < 4.0e9 ? (unsigned)n : 0xffffffffu;
  return b;
}

}  // namespace nodes
}  // namespace xs
