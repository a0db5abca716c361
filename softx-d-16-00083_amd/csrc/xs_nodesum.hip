// H3 for histograms: pair sums S_p(q) = sum_k h_p[k] sin(q r_k)/(q r_k + 1e-8),
// r_k = (k + 1/2) bin, over Chebyshev nodes of groups of bins.
//
// On a group of bins that spans 4 c / Q (|q| <= Q), sin(q r)/(q r) is its
// Chebyshev interpolant through K = 64 points to FP64 rounding for c = 14.2
// (2 c^K / K! = 1e-15, see xs_nodes.h), so the group's counts act through 64
// node weights, W_m = sum_k h[k] L_m(t_k): at 0.005 A and 25 1/A, 454 bins become
// 64 nodes.  Then S = W F with F[node][q] = sin(q r)(y - (1e-8/(q bin)) y^2),
// y = bin / r, is a matrix product, of 16 histograms x 16 q x 4 nodes per
// v_mfma_f64_16x16x4.
//   tables    max |q| and with it the bins per group; L_m(t_k) of a group (one
//             table for all); y of the nodes; S cleared
//   weights   W of a group of 16 histograms: the product H L, on the same
//             instruction, the bins shared by 8 waves
//   sums      the product W F.  A wave owns 16 q and up to 8 tiles of 16
//             histograms; it forms F in registers: sin(q (r_g + d_m)) from
//             sin, cos(q r_g), turned on from group to group, and the 64
//             sin, cos(q d_m), made once (two operations), and two more for the
//             weight of the denominator
//   few       the same for up to 8 histograms, with groups as the rows
// 3 histograms of 97,251 bins x 4,096 q: tables 9 us, weights 15, few 25 (a term per
// bin and q, a rotation each: 222).  768 x 16,384 bins x 8,192 q: tables 14, weights
// 74, sums 493, of which the matrix instructions are 360 at the 67 TFLOP/s that a
// large product reaches.
// Group 0 reaches r = 0, where 1/r has no series: it carries h / r and sin(q r)
// alone, and group 1 carries h / r^2 of the same bins for the 1e-8 term.
// Where the bins are too wide for groups of more than 96 (Q bin above ~0.6) each
// bin is a node: the same product without a gain from the groups, for which one
// histogram of 7,303 bins x 1,257 q takes 20 us (a rotation per bin and q: 66).
#include <algorithm>
#include <cmath>

#include "xs_nodes.h"
#include "xs_nodesum.h"
#include "xs_sincos.h"

namespace xs {
namespace nodesum {

typedef double double4v __attribute__((ext_vector_type(4)));

struct PlanArgs {
  const double *q;
  unsigned nq;
  double bin, c;
  Row *rows;  // tables of ntypes histograms of nhist bins, or nullptr
  uint32_t *nmax;
  unsigned ntypes, nhist, ntiles;
  unsigned limit;  // bins of a group at most
};

// Bins per group for |q| <= Q: the largest B with Q B bin / 4 <= c, at most the limit.
// Every thread of the work group gets the plan.
__device__ Plan make_plan(const PlanArgs &A) {
  __shared__ double sh[16];
  double m = 0.0;
  for (unsigned i = threadIdx.x; i < A.nq; i += blockDim.x) m = fmax(m, fabs(A.q[i]));
  for (int w = 32; w > 0; w >>= 1) m = fmax(m, __shfl_xor(m, w, 64));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  for (unsigned i = 0; i < blockDim.x / 64; ++i) m = fmax(m, sh[i]);
  const double b = floor(4.0 * A.c / (m * A.bin));
  // (m = 0: infinite; an infinite q: 0)
  const unsigned bins = b > (double)A.limit ? A.limit : b > 0.0 ? (unsigned)b : 0u;
  Plan P;
  P.compress = bins > kNodes + kNodes / 2;
  P.bins = P.compress ? bins : kNodes;
  return P;
}

__device__ void store_plan(const PlanArgs &A, const Plan &P, Plan *plan) {
  if (threadIdx.x == 0) *plan = P;
  for (unsigned i = threadIdx.x; A.rows && i < A.ntiles * kRows; i += blockDim.x) {
    A.rows[i] = Row{i < A.ntypes ? (unsigned long long)i * A.nhist : 0ull,
                    i < A.ntypes ? A.nhist : 0u, i};
    if (i < A.ntiles) A.nmax[i] = A.nhist;
  }
}

// One work group, where nq is too large for every one of tables_kernel's to read.
constexpr unsigned kPlanAll = 16384;
__global__ __launch_bounds__(1024) void plan_kernel(PlanArgs A, Plan *__restrict__ plan) {
  store_plan(A, make_plan(A), plan);
}

// cos(2 pi n / 256), n < 256: T_j(x_m) = cos(j pi (m + 1/2) / 64) is entry
// j (2 m + 1) mod 256.
__device__ __forceinline__ void cos_table(double *tab) {
  for (unsigned n = threadIdx.x; n < 4 * kNodes; n += blockDim.x) {
    double s, c;
    sincos_2pi((double)n / (4.0 * kNodes), &s, &c);
    tab[n] = c;
  }
}

// Offset of node m from its group's centre, in bins.
__device__ __forceinline__ double node_offset(const Plan &P, unsigned m) {
  if (!P.compress) return (double)m - 0.5 * (kNodes - 1);
  double s, c;
  sincos_2pi((double)(2 * m + 1) / (4.0 * kNodes), &s, &c);
  return 0.5 * (double)P.bins * c;
}

// Group g: the bins it stands for (groups 0 and 1: the first ones).
__device__ __forceinline__ unsigned group_bins(unsigned g) { return g < 2 ? 0u : g - 1; }

// The plan (its own copy in each work group), then: L[k][m] (4 k a work group,
// thread (m, k)); node[g 64 + m] = factors of 1 and of -1e-8/(q bin) in the node's
// F (the next (group_cap + 3) / 4 work groups, 4 groups each); the others clear S.
__global__ __launch_bounds__(4 * kNodes) void tables_kernel(PlanArgs A, Plan *__restrict__ plan,
                                                            unsigned group_cap,
                                                            double *__restrict__ L,
                                                            double2 *__restrict__ node,
                                                            double *__restrict__ S, size_t ssize) {
  __shared__ double tab[4 * kNodes];
  Plan P;
  if (A.nq > kPlanAll) {
    P = *plan;
  } else {
    P = make_plan(A);
    if (blockIdx.x == 0) store_plan(A, P, plan);
  }
  const unsigned m = threadIdx.x % kNodes, part = threadIdx.x / kNodes;
  const unsigned node0 = (A.limit + 3) / 4, zero0 = node0 + (group_cap + 3) / 4;
  if (blockIdx.x >= zero0) {
    for (size_t i = (blockIdx.x - zero0) * (size_t)blockDim.x + threadIdx.x; i < ssize;
         i += (size_t)(gridDim.x - zero0) * blockDim.x)
      S[i] = 0.0;
    return;
  }
  if (blockIdx.x >= node0) {
    const unsigned g = (blockIdx.x - node0) * 4 + part;
    if (g >= group_cap) return;
    const double r = ((double)group_bins(g) + 0.5) * (double)P.bins + node_offset(P, m);
    const double y = 1.0 / r;
    double2 v = make_double2(y, y * y);
    if (P.compress && g == 0) v = make_double2(1.0, 0.0);
    if (P.compress && g == 1) v = make_double2(0.0, 1.0);
    node[(size_t)g * kNodes + m] = v;
    return;
  }
  if (!P.compress || blockIdx.x * 4 >= P.bins) return;
  cos_table(tab);
  __syncthreads();
  const unsigned k = blockIdx.x * 4 + part;
  if (k >= P.bins) return;
  const double t = (2.0 * k + 1.0) / (double)P.bins - 1.0;
  double t0 = 1.0, t1 = t, sum = 0.0;
  for (unsigned j = 1; j < kNodes; ++j) {
    sum = fma(t1, tab[(j * (2 * m + 1)) % (4 * kNodes)], sum);
    const double tn = fma(2.0 * t, t1, -t0);
    t0 = t1;
    t1 = tn;
  }
  L[(size_t)k * kNodes + m] = (1.0 + 2.0 * sum) / kNodes;
}

constexpr int kWaves = 8;  // of weights_kernel

// The weights w[node][16 rows] of a group in the form that few_kernel reads: for
// m < 32 the sums w_m y_m + w_{63-m} y_{63-m} and differences, and those of y^2, as
// [row][group / 16][y, y^2][sum, difference][m / 4][16 (m mod 4) + group mod 16].
__device__ __forceinline__ void few_weights(const double *w, const double2 *node, unsigned nrows,
                                            unsigned g, unsigned ngroups, double *__restrict__ W) {
  for (unsigned i = threadIdx.x; i < nrows * 2 * kNodes; i += 64 * kWaves) {
    const unsigned row = i / (2 * kNodes), part = i / (kNodes / 2) % 4, m = i % (kNodes / 2);
    const double2 ya = node[m], yb = node[kNodes - 1 - m];
    const double a = w[m * kRows + row] * (part < 2 ? ya.x : ya.y),
                 b = w[(kNodes - 1 - m) * kRows + row] * (part < 2 ? yb.x : yb.y);
    W[(((size_t)row * (ngroups / 16) + g / 16) * 32 + part * 8 + m / 4) * 64 + m % 4 * 16 + g % 16] =
        part & 1 ? a - b : a + b;
  }
}

// W[tile][group][node][16 rows], or few_weights' form for `few` rows; one work
// group per group (x) and tile (y).  Bound by the latency of the loads of L (L2) and
// the counts: 120 registers leave two work groups a CU (counts of 32 bins ahead, 144
// registers and one a CU: 92 us for 768 histograms of 16,384 bins; 16 ahead: 74).
__global__ __launch_bounds__(64 * kWaves, 4) void weights_kernel(
    const unsigned long long *__restrict__ hist, const Row *__restrict__ rows,
    const uint32_t *__restrict__ nmax, unsigned tile0, unsigned group0, const Plan *__restrict__ plan,
    const double *__restrict__ L, const double2 *__restrict__ node, unsigned few,
    unsigned ct, double *__restrict__ W) {
  __shared__ double red[kWaves][kNodes * kRows];
  const Plan P = *plan;
  const unsigned g = group0 + blockIdx.x, tile = tile0 + blockIdx.y;
  // zeros up to the longest of the ct tiles that a wave of sums_kernel takes at once
  // (few_kernel: 16 groups)
  const unsigned ng = groups_for(nmax[few ? tile : tile - blockIdx.y % ct], P.bins);
  if (g >= (few ? align_groups(ng) : ng)) return;
  double *out = W + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * kNodes * kRows;
  const unsigned first = group_bins(g) * P.bins;
  if (!P.compress) {
    for (unsigned i = threadIdx.x; i < kNodes * kRows; i += 64 * kWaves) {
      const Row r = rows[tile * kRows + i % kRows];
      const unsigned k = first + i / kRows;
      const double v = g != 1 && k < r.nhist ? (double)hist[r.hist_off + k] : 0.0;
      if (few)
        red[0][i] = v;
      else
        out[i] = v;
    }
    if (few) {
      __syncthreads();
      few_weights(red[0], node + (size_t)g * kNodes, few, blockIdx.x, gridDim.x, W);
    }
    return;
  }
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kc = lane >> 4;
  const Row r = rows[tile * kRows + col];
  double4v acc[4];
  for (int t = 0; t < 4; ++t) acc[t] = (double4v){0.0, 0.0, 0.0, 0.0};
  // each wave a contiguous eighth of the bins; the counts of 16 bins and L of 8
  // are loaded ahead
  const unsigned per = (P.bins + 4 * kWaves - 1) / (4 * kWaves) * 4;
  const unsigned begin = wave * per, end = first < nmax[tile] ? min(P.bins, begin + per) : 0u;
  unsigned long long n[2][4];
  double l[2][2][4];
  const unsigned long long *hrow = hist + r.hist_off + first;
  const unsigned kend = first < r.nhist ? min(end, r.nhist - first) : 0u;
  auto load_counts = [&](unsigned k0, int b) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const unsigned k = k0 + 4 * u + kc;
      n[b][u] = k < kend ? hrow[k] : 0ull;
    }
  };
  auto load_L = [&](unsigned k0, int b) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const double *lp = L + (size_t)min(k0 + 4 * u + kc, P.bins - 1) * kNodes + col;
#pragma unroll
      for (int t = 0; t < 4; ++t) l[b][u][t] = lp[16 * t];
    }
  };
  load_counts(begin, 0);
  load_L(begin, 0);
#pragma unroll 1
  for (unsigned k0 = begin; k0 < end; k0 += 32)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      load_counts(k0 + 16 * h + 16, h ^ 1);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const unsigned kb = k0 + 16 * h + 8 * b;
        if (kb >= end) break;
        load_L(kb + 8, (b & 1) ^ 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const unsigned long long nu = n[h][2 * b + u];
          double x = (double)nu;
          if (g < 2) {
            const double y = 1.0 / ((double)(first + kb + 4 * u + kc) + 0.5);
            x *= g ? y * y : y;
          }
#pragma unroll
          for (int t = 0; t < 4; ++t)
            acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, l[b & 1][u][t], acc[t], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  // row (lane >> 4) + 4 r of the product is a histogram, column lane & 15 of
  // tile t node 16 t + column
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][(16 * t + col) * kRows + kc + 4 * i] = acc[t][i];
  __syncthreads();
  for (unsigned i = threadIdx.x; i < kNodes * kRows; i += 64 * kWaves) {
    double v = 0.0;
    for (int w = 0; w < kWaves; ++w) v += red[w][i];
    if (few)
      red[0][i] = v;
    else
      out[i] = v;
  }
  if (few) {
    __syncthreads();
    few_weights(red[0], node + (size_t)g * kNodes, few, blockIdx.x, gridDim.x, W);
  }
}

// S += W F.  Grid (blocks of 64 q, groups of CT tiles, shares of the groups of
// bins); a wave has 16 q.
constexpr unsigned kReseed = 8;  // groups between fresh sin, cos(q r_g)
template <int CT>
__global__ __launch_bounds__(256, CT > 1 ? 3 : 4) void sums_kernel(const double *__restrict__ W,
                                                   const Row *__restrict__ rows,
                                                   const uint32_t *__restrict__ nmax,
                                                   unsigned tile0, unsigned ntiles,
                                                   unsigned group0, unsigned ngroups, unsigned nrows,
                                                   const Plan *__restrict__ plan,
                                                   const double2 *__restrict__ node, double bin,
                                                   const double *__restrict__ q, unsigned nq,
                                                   double *__restrict__ S, int add) {
  __shared__ double2 turn[4][kNodes / 2][16];  // sin, cos of q d_m; d_{63-m} = -d_m
  const Plan P = *plan;
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kc = lane >> 4;
  const unsigned iq = blockIdx.x * 64 + wave * 16 + col;
  const double qv = q[min(iq, nq - 1)];
  constexpr double kTwoPi = 6.283185307179586476925286766559;
  const double turns = qv * bin / kTwoPi;  // phase step per bin, in turns
  const double eq = qv == 0.0 ? 0.0 : 1e-8 / (qv * bin);
  for (unsigned m = kc; m < kNodes / 2; m += 4) {
    double s, c;
    sincos_2pi(node_offset(P, m) * turns, &s, &c);
    turn[wave][m][col] = make_double2(s, c);
  }
  __syncthreads();
  const unsigned t0 = blockIdx.y * CT, nt = min((unsigned)CT, ntiles - t0);
  // groups of the longest tile (the first: the tiles are in order of length)
  const unsigned ge = min(groups_for(nmax[tile0 + t0], P.bins), group0 + ngroups);
  const unsigned ng = ge > group0 ? ge - group0 : 0u;
  const unsigned g0 = group0 + (unsigned)((unsigned long long)ng * blockIdx.z / gridDim.z);
  const unsigned g1 = group0 + (unsigned)((unsigned long long)ng * (blockIdx.z + 1) / gridDim.z);
  // (few tiles: two sums a tile, so that no product waits for the last one)
  constexpr int kHalves = CT <= 2 ? 2 : 1;
  double4v acc[kHalves][CT];
#pragma unroll
  for (int h = 0; h < kHalves; ++h)
#pragma unroll
    for (int t = 0; t < CT; ++t) acc[h][t] = (double4v){0.0, 0.0, 0.0, 0.0};
  double hs, hc;  // a turn of one group
  sincos_2pi((double)P.bins * turns, &hs, &hc);
  double gs = 0.0, gc = 1.0;
  const size_t tile_size = (size_t)ngroups * kNodes * kRows;
  // lane's weights: row col of node 4 step + kc.  kSteps steps' weights and node
  // factors are loaded ahead of the products of the steps before them (the
  // compiler would load each where it is used; sched_barrier keeps it from that)
  constexpr int kSteps = CT == 1 ? 4 : 8 / CT;
  const double *w0 = W + (size_t)t0 * tile_size;
  double a[2][kSteps][CT];
  double2 c[2][kSteps];
  auto load = [&](unsigned g, int i, int b) {
    const double *wg = w0 + (size_t)(g - group0) * kNodes * kRows + i * kSteps * 64;
    const double2 *nd = node + (size_t)g * kNodes + 4 * i * kSteps;
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
#pragma unroll
      for (int t = 0; t < CT; ++t) a[b][u][t] = (wg + min((unsigned)t, nt - 1) * tile_size + u * 64)[lane];
      c[b][u] = (nd + 4 * u)[kc];
    }
  };
  if (g0 < g1) load(g0, 0, 0);
  for (unsigned g = g0; g < g1; ++g) {
    if (g == g0 || g <= 2 || (g - g0) % kReseed == 0) {
      sincos_2pi(((double)group_bins(g) + 0.5) * (double)P.bins * turns, &gs, &gc);
    } else {
      const double s = fma(gs, hc, gc * hs);
      gc = fma(gc, hc, -(gs * hs));
      gs = s;
    }
    constexpr int kBatches = (int)kNodes / 4 / kSteps;
#pragma unroll 1
    for (int i0 = 0; i0 < kBatches; i0 += 2)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int i = i0 + b;
        const bool last = i == kBatches - 1;
        load(last ? min(g + 1, g1 - 1) : g, last ? 0 : i + 1, b ^ 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
          const unsigned st = i * kSteps + u;
          const bool up = st < kNodes / 8;
          const double2 d = turn[wave][up ? 4 * st + kc : kNodes - 1 - 4 * st - kc][col];
          const double x = gc * d.x;
          const double f = fma(gs, d.y, up ? x : -x) * fma(-eq, c[b][u].y, c[b][u].x);
#pragma unroll
          for (int t = 0; t < CT; ++t)
            acc[u % kHalves][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[b][u][t], f,
                                                                       acc[u % kHalves][t], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
  }
  if (iq >= nq) return;
  const double scale = qv == 0.0 ? 0.0 : 1.0 / (qv * bin);
#pragma unroll
  for (int t = 0; t < CT; ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned row = (tile0 + t0 + t) * kRows + kc + 4 * i;
      if (t >= (int)nt || row >= nrows) continue;
      double *p = S + (size_t)rows[row].srow * nq + iq;
      double v = acc[0][t][i];
      if (kHalves > 1) v += acc[kHalves - 1][t][i];
      v = qv == 0.0 ? 0.0 : v * scale;
      if (add)
        atomicAdd(p, v);
      else
        *p = v;
    }
  }
}

// S += W F of a few histograms: the sines of a group's nodes are
// sin(q (r_g + d_m)) = sin(q r_g) cos(q d_m) + cos(q r_g) sin(q d_m), so the sums
// over the 64 nodes are products with one table of 32 cosines and 32 sines per q,
// kept in registers, whose other side is 16 groups of ONE histogram: no row of
// the product is idle, and a sine is formed once a group, not once a node.  The
// price is a second product for the weights of the denominator's 1e-8, which the
// kernel above folds into F for two operations a node and 16 histograms.  97,251
// bins x 4,096 q, whole call: 1 histogram 37 us, 8 72, and by the kernel above 9 to
// 16 91 (its 16 rows cost the same for any number): the lines would meet at 12, the
// weights' memory of a tile holds 8.  Bound by the latency of a wave's few tiles
// (25 us of which 10 are matrix instructions); weights loaded where they are used
// 46.
// Grid (blocks of 64 q, histograms, shares of the groups); a wave has 16 q.
__global__ __launch_bounds__(256) void few_kernel(const double *__restrict__ W,
                                                  const Row *__restrict__ rows, unsigned group0,
                                                  unsigned ngroups, const Plan *__restrict__ plan,
                                                  double bin, const double *__restrict__ q,
                                                  unsigned nq, double *__restrict__ S, int add) {
  const Plan P = *plan;
  const Row r = rows[blockIdx.y];
  const unsigned ge = min(align_groups(groups_for(r.nhist, P.bins)), group0 + ngroups);
  const unsigned nt = ge > group0 ? (ge - group0) / 16 : 0u;
  const unsigned t0 = (unsigned)((unsigned long long)nt * blockIdx.z / gridDim.z);
  const unsigned t1 = (unsigned)((unsigned long long)nt * (blockIdx.z + 1) / gridDim.z);
  if (t0 == t1 && add) return;
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kc = lane >> 4;
  const unsigned iq = blockIdx.x * 64 + wave * 16 + col;
  const double qv = q[min(iq, nq - 1)];
  constexpr double kTwoPi = 6.283185307179586476925286766559;
  const double turns = qv * bin / kTwoPi;  // phase step per bin, in turns
  const double eq = qv == 0.0 ? 0.0 : 1e-8 / (qv * bin);
  // column col = q, row kc of step st = node 4 st + kc
  double ct[8], sn[8];
#pragma unroll
  for (int st = 0; st < 8; ++st) sincos_2pi(node_offset(P, 4 * st + kc) * turns, &sn[st], &ct[st]);
  double hs, hc;  // a turn of four groups
  sincos_2pi(4.0 * (double)P.bins * turns, &hs, &hc);
  double sum = 0.0, sum1 = 0.0;
  // two steps' weights ahead of the products (the compiler would load each where
  // it is used; sched_barrier keeps it from that)
  const double *w0 = W + (size_t)blockIdx.y * (ngroups / 16) * 32 * 64 + lane;
  double a[2][2][4];
  auto load = [&](unsigned t, int c, int b) {
    const double *w = w0 + (size_t)t * 32 * 64 + c * 2 * 64;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) a[b][u][i] = w[(i * 8 + u) * 64];
  };
  if (t0 < t1) load(t0, 0, 0);
  for (unsigned t = t0; t < t1; ++t) {
    double4v p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = (double4v){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      load(c == 3 ? min(t + 1, t1 - 1) : t, (c + 1) & 3, (c + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          p[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[c & 1][u][i],
                                                      i & 1 ? sn[2 * c + u] : ct[2 * c + u], p[i], 0,
                                                      0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the lane's rows: groups g + 4 i of the 16
    const unsigned g = group0 + 16 * t + kc;
    double gs, gc;
    sincos_2pi(((double)(g ? g - 1 : 0u) + 0.5) * (double)P.bins * turns, &gs, &gc);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sum = fma(gs, p[0][i], fma(gc, p[1][i], sum));
      sum1 = fma(gs, p[2][i], fma(gc, p[3][i], sum1));
      if (i == 0 && g == 0) {  // group 4 is three groups' turn from group 1
        sincos_2pi(3.5 * (double)P.bins * turns, &gs, &gc);
      } else {
        const double s = fma(gs, hc, gc * hs);
        gc = fma(gc, hc, -(gs * hs));
        gs = s;
      }
    }
  }
  double v = fma(-eq, sum1, sum);
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  if (iq >= nq || kc != 0) return;
  v = qv == 0.0 ? 0.0 : v / (qv * bin);
  double *out = S + (size_t)r.srow * nq + iq;
  if (add)
    atomicAdd(out, v);
  else
    *out = v;
}

Layout layout(unsigned ntiles, unsigned nhist_max, size_t budget) {
  Layout L{};
  L.ntiles = ntiles;
  L.nhist_max = nhist_max;
  L.group_cap = align_groups(groups_for(nhist_max, kNodes));
  const size_t group = (size_t)kNodes * kRows * 8;
  L.groups_at_once = (unsigned)std::min<size_t>(L.group_cap, std::max<size_t>(16, budget / group / 16 * 16));
  L.tiles_at_once = (unsigned)std::min<size_t>(
      ntiles, std::max<size_t>(1, budget / (group * L.groups_at_once)));
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t p = at;
    at = align_up(at + bytes, 256);
    return p;
  };
  L.plan = take(sizeof(Plan));
  L.rows = take((size_t)ntiles * kRows * sizeof(Row));
  L.nmax = take((size_t)ntiles * 4);
  L.lagrange = take((size_t)kMaxBins * kNodes * 8);
  L.node = take((size_t)L.group_cap * kNodes * 16);
  L.weights = take(group * L.groups_at_once * L.tiles_at_once);
  L.total = at;
  return L;
}

// Bins per group at most.  The weights of a group are one work group's, so large groups
// take time where there are few (4,096 bins: 85 us for one histogram of 3,000 bins that
// 15 smaller groups do in 30), and for few_kernel 16 groups cost as much as one.  Where
// the products are the larger part, only the bound of the tables.
static unsigned group_limit(unsigned nrows, unsigned nq, unsigned nhist_max) {
  if (nrows > kFew && (size_t)nrows * nq > 131072) return kMaxBins;
  return std::min(1024u, std::max(kNodes + kNodes / 2 + 1, (nhist_max + 13) / 14));
}

static int tables(xs_ctx *ctx, const Tables &T, unsigned limit, double bin, const double *q, unsigned nq,
                  double *S, size_t ssize) {
  const Layout &L = T.L;
  hipStream_t st = ctx->stream;
  // 2 c^64 / 64! = 1e-15
  const double c = nodes::reach((int)kNodes, 1e-15);
  const PlanArgs A{q, nq, bin, c, T.ntypes ? T.at<Row>(L.rows) : nullptr,
                   T.ntypes ? T.at<uint32_t>(L.nmax) : nullptr, T.ntypes, T.nhist, L.ntiles, limit};
  if (nq > kPlanAll)
    hipLaunchKernelGGL(plan_kernel, dim3(1), dim3(1024), 0, st, A, T.at<Plan>(L.plan));
  const unsigned zb = (unsigned)std::min<size_t>((ssize + 1023) / 1024, 1024);
  hipLaunchKernelGGL(tables_kernel, dim3((limit + 3) / 4 + (L.group_cap + 3) / 4 + zb), dim3(4 * kNodes), 0,
                     st, A, T.at<Plan>(L.plan), L.group_cap, T.at<double>(L.lagrange),
                     T.at<double2>(L.node), S, ssize);
  XS_HIP_CHECK(hipGetLastError());
  return XS_OK;
}

// As many tiles a wave as leave two work groups a CU, so that a sine serves more of
// them.
static unsigned tiles_a_wave(const xs_ctx *ctx, unsigned ntiles, unsigned nq) {
  for (unsigned c : {8u, 4u, 2u})
    if (ntiles >= c && (size_t)((nq + 63) / 64) * ((ntiles + c - 1) / c) >= 2 * (size_t)ctx->cu_count)
      return c;
  return 1;
}

static int weights(xs_ctx *ctx, const Tables &T, const unsigned long long *hist, unsigned nrows,
                   unsigned nq, unsigned tile0, unsigned ntiles, unsigned group0, unsigned ngroups) {
  const Layout &L = T.L;
  hipLaunchKernelGGL(weights_kernel, dim3(ngroups, ntiles), dim3(64 * kWaves), 0, ctx->stream, hist,
                     T.rows(), T.nmax(), tile0, group0, T.at<Plan>(L.plan), T.at<double>(L.lagrange),
                     T.at<double2>(L.node), nrows <= kFew ? nrows : 0u,
                     tiles_a_wave(ctx, ntiles, nq), T.at<double>(L.weights));
  XS_HIP_CHECK(hipGetLastError());
  return XS_OK;
}

static int sums(xs_ctx *ctx, const Tables &T, unsigned tile0, unsigned ntiles, unsigned group0,
                unsigned ngroups, unsigned nrows, double bin, const double *q, unsigned nq, double *S) {
  const Layout &L = T.L;
  const unsigned qb = (nq + 63) / 64;
  if (nrows <= kFew) {
    const unsigned z = std::min<unsigned>(ngroups / 16,
                                          std::max(1u, 4 * (unsigned)ctx->cu_count / (qb * nrows)));
    hipLaunchKernelGGL(few_kernel, dim3(qb, nrows, z), dim3(256), 0, ctx->stream,
                       T.at<double>(L.weights), T.rows(), group0, ngroups, T.at<Plan>(L.plan), bin, q,
                       nq, S, z > 1 || ngroups < L.group_cap);
    XS_HIP_CHECK(hipGetLastError());
    return XS_OK;
  }
  const unsigned ct = tiles_a_wave(ctx, ntiles, nq);
  const unsigned tg = (ntiles + ct - 1) / ct;
  // shares of the groups of bins where the chip would not be full
  unsigned z = 1;
  while (z < 32 && (size_t)qb * tg * z < 4 * (size_t)ctx->cu_count && 4 * z <= ngroups) z *= 2;
  int add = z > 1 || ngroups < L.group_cap;
  const dim3 grid(qb, tg, z);
  const void *k[4] = {reinterpret_cast<const void *>(&sums_kernel<1>),
                      reinterpret_cast<const void *>(&sums_kernel<2>),
                      reinterpret_cast<const void *>(&sums_kernel<4>),
                      reinterpret_cast<const void *>(&sums_kernel<8>)};
  const double *W = T.at<double>(L.weights);
  const Row *rows = T.rows();
  const uint32_t *nmax = T.nmax();
  const Plan *plan = T.at<Plan>(L.plan);
  const double2 *node = T.at<double2>(L.node);
  void *args[] = {&W,      &rows, &nmax, &tile0, &ntiles, &group0, &ngroups, &nrows,
                  &plan,   &node, &bin,  &q,     &nq,     &S,      &add};
  XS_HIP_CHECK(hipLaunchKernel(k[ct == 1 ? 0 : ct == 2 ? 1 : ct == 4 ? 2 : 3], grid, dim3(256), args, 0,
                               ctx->stream));
  return XS_OK;
}

int run(xs_ctx *ctx, const Tables &T, const unsigned long long *hist, unsigned nrows, double bin,
        const double *q, unsigned nq, double *S) {
  const Layout &L = T.L;
  XS_TRY(tables(ctx, T, group_limit(nrows, nq, L.nhist_max), bin, q, nq, S, (size_t)nrows * nq));
  for (unsigned t = 0; t < L.ntiles; t += L.tiles_at_once)
    for (unsigned g = 0; g < L.group_cap; g += L.groups_at_once) {
      const unsigned nt = std::min(L.tiles_at_once, L.ntiles - t),
                     ng = std::min(L.groups_at_once, L.group_cap - g);
      XS_TRY(weights(ctx, T, hist, nrows, nq, t, nt, g, ng));
      XS_TRY(sums(ctx, T, t, nt, g, ng, nrows, bin, q, nq, S));
    }
  return XS_OK;
}

}  // namespace nodesum
}  // namespace xs
