// H5/H6 through Chebyshev moments of the pair distances (xs_nodes.h).
//
// The direct Debye sums cost pairs x nq terms; here each pair costs its
// distance and K moments, and the q mesh meets only nb x K nodes per row of S
// (a pair type, or a pair type and block pair).  Three kernels:
//   moments  one work group per run of 64 x 64-atom tile pairs of one segment
//            pair; the moments of all bins live in LDS.  T_0 is a uint32
//            count, T_k (k >= 1) a 64-bit fixed-point sum: T_k 2^s + 1.5 2^52
//            in one FMA leaves the integer in the low mantissa bits, so the
//            raw bits are added with ds_add_u64 and count x bits(1.5 2^52) is
//            subtracted once at the end.  s is as large as the run's pairs
//            allow (62 - log2 of them, 48 at most), so the sum cannot overflow
//            and a moment is rounded at 2^-(s+1) per pair; integer sums do
//            not depend on their order.  ds_add_u64 on random bins takes 11.4
//            CU cycles a wave, ds_add_u32 6.2, ds_add_f64 21.7 (measured;
//            an odd 8-byte stride between bins, an even one takes 3 times as
//            long): the kernel is bound by these LDS atomics, its ~45 VALU
//            instructions a pair run beside them.
//   reduce   adds up the runs' slabs per row, in run order.
//   eval     node weights from the moments (a K-point cosine transform), then
//            sum over nodes of weight x f_q(node), one q per lane, up to 8
//            rows at once so that a sine serves all of them.
// Bin 0 reaches r = 0, where the e/r^2 part of f_q has no series: its pairs
// also go, weighted with 1/r, into a bin of their own that carries this part
// (and bin 0 carries the 1/r part alone).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "xs_debye_moments.h"
#include "xs_internal.h"
#include "xs_sincos.h"

namespace xs {
namespace debye {

constexpr int kMTile = 64;          // atoms per tile: one per lane
constexpr int kMBlock = 1024;
constexpr size_t kMLds = 160000;    // of the CU's 163,840 bytes
constexpr double kMagic = 6755399441055744.0;            // 1.5 * 2^52
constexpr unsigned long long kMagicBits = 0x4338000000000000ull;
constexpr double kTwoPi = 6.283185307179586476925286766559;

// A run of tile pairs of segments A and B: items first .. first + count,
// an item being a tile pair's share of jr J atoms.
struct Run {
  uint32_t first, count, offA, cntA, offB, cntB, diag, pad;
};

static size_t lds_bytes(unsigned nb, int K) {
  return (size_t)nb * (K - 1) * 8 + align_up((size_t)nb * 4, 8) + (size_t)K * 8;
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  const unsigned long long u = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)u, lane);
  const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
  return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}

// sqrt(s) to within an ulp or two for normal s: v_rsq_f64, one Goldschmidt
// step and one residual correction (the IEEE root's range scaling and its
// last-bit fix are not needed: an ulp of r is the rounding of its inputs).
__device__ __forceinline__ double root(double s) {
  const double y = __builtin_amdgcn_rsq(s);
  double g = s * y, h = 0.5 * y;
  const double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  return fma(fma(-g, g, s), h, g);
}

template <int K>
__global__ __launch_bounds__(kMBlock) void moments_kernel(
    const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
    const Run *__restrict__ runs, double *__restrict__ slabs, double inv_h, unsigned nb,
    double scale, double unscale, unsigned sub_shift) {
  extern __shared__ unsigned long long mom[];  // [nb][K - 1], K - 1 odd
  uint32_t *cnt = reinterpret_cast<uint32_t *>(mom + (size_t)nb * (K - 1));
  double *near = reinterpret_cast<double *>(cnt + ((nb + 1) & ~1u));
  static_assert(K % 2 == 0, "odd stride between bins");
  const unsigned words = nb * (K - 1) + (nb + 1) / 2 + K;
  for (unsigned i = threadIdx.x; i < words; i += kMBlock) mom[i] = 0;
  const Run run = runs[blockIdx.x];
  const unsigned lane = threadIdx.x & 63;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned TA = (run.cntA + kMTile - 1) / kMTile, TB = (run.cntB + kMTile - 1) / kMTile;
  const unsigned jr = kMTile >> sub_shift;
  __syncthreads();
  for (unsigned m = run.first + wave; m < run.first + run.count; m += kMBlock / 64) {
    const unsigned sub = m & ((1u << sub_shift) - 1), tp = m >> sub_shift;
    unsigned ti, tj;
    if (run.diag) {
      // row ti holds the J tiles ti..TB-1; rows before it c(ti) pairs
      const double T2 = 2.0 * (double)TB + 1.0;
      const double g = floor(0.5 * (T2 - sqrt(fmax(T2 * T2 - 8.0 * (double)tp, 0.0))));
      uint64_t i = g < 0.0 ? 0 : (uint64_t)g;
      if (i >= TB) i = TB - 1;
      auto c = [TB](uint64_t v) { return v * TB - v * (v - 1) / 2; };
      while (i > 0 && c(i) > tp) --i;
      while (i + 1 < TB && c(i + 1) <= tp) ++i;
      ti = __builtin_amdgcn_readfirstlane((unsigned)i);
      tj = __builtin_amdgcn_readfirstlane((unsigned)(i + (tp - c(i))));
    } else {
      ti = tp / TB;
      tj = tp % TB;
    }
    // a tile is every TA-th (TB-th) atom: the lanes' distances to a J atom then
    // spread over the bins
    const unsigned ia = ti + lane * TA, ja = tj + lane * TB;
    const size_t gi = (size_t)run.offA + min(ia, run.cntA - 1);
    const size_t gj = (size_t)run.offB + min(ja, run.cntB - 1);
    const double xi = x[gi], yi = y[gi], zi = z[gi];
    const double xj = x[gj], yj = y[gj], zj = z[gj];
    // J atoms this lane pairs with: all, or those after its own atom
    const unsigned jmin = ia >= run.cntA ? 0xffffffffu
                          : (run.diag && ti == tj) ? lane + 1 : 0u;
    const unsigned j1 = min(sub * jr + jr, (run.cntB - tj + TB - 1) / TB);
    for (unsigned j = sub * jr; j < j1; ++j) {
      const double dx = xi - lane_value(xj, j), dy = yi - lane_value(yj, j),
                   dz = zi - lane_value(zj, j);
      const double s = fma(dx, dx, fma(dy, dy, dz * dz));
      if (j >= jmin && s > 0.0) {
        const double r = root(s);
        const double u = r * inv_h;
        const unsigned b = min((unsigned)u, nb - 1);
        const double t = fma(2.0, __builtin_amdgcn_fract(u), -1.0);
        __hip_atomic_fetch_add(&cnt[b], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        unsigned long long *p = mom + b * (K - 1);
        double tp0 = 1.0, tp1 = t;
        const double t2 = t + t;
#pragma unroll
        for (int k = 1; k < K; ++k) {
          const unsigned long long v = __double_as_longlong(fma(tp1, scale, kMagic));
          __hip_atomic_fetch_add(p + k - 1, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          const double tn = fma(t2, tp1, -tp0);
          tp0 = tp1;
          tp1 = tn;
        }
        if (b == 0) {
          double a0 = 1.0, a1 = t;
          const double ir = 1.0 / r;
          for (int k = 0; k < K; ++k) {
            __hip_atomic_fetch_add(near + k, a0 * ir, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            const double an = fma(t2, a1, -a0);
            a0 = a1;
            a1 = an;
          }
        }
      }
    }
  }
  __syncthreads();
  double *slab = slabs + (size_t)blockIdx.x * ((size_t)nb + 1) * K;
  for (unsigned e = threadIdx.x; e < nb * K; e += kMBlock) {
    const unsigned b = e / K, k = e % K;
    const unsigned long long n = cnt[b];
    double v = (double)n;
    if (k) v = (double)(long long)(mom[b * (K - 1) + k - 1] - n * kMagicBits) * unscale;
    slab[e] = v;
  }
  if (threadIdx.x < K) slab[(size_t)nb * K + threadIdx.x] = near[threadIdx.x];
}

// M[row][e] = sum of the row's slabs; 64 entries and 16 shares of the slabs
// per work group.
__global__ __launch_bounds__(1024) void reduce_kernel(const double *__restrict__ slabs,
                                                      const uint32_t *__restrict__ row_run,
                                                      unsigned entries, double *__restrict__ M) {
  __shared__ double part[16][64];
  const unsigned row = blockIdx.y, e = blockIdx.x * 64 + (threadIdx.x & 63), g = threadIdx.x >> 6;
  const unsigned r1 = row_run[row + 1];
  double a = 0.0;
  if (e < entries)
    for (unsigned r = row_run[row] + g; r < r1; r += 16) a += slabs[(size_t)r * entries + e];
  part[g][threadIdx.x & 63] = a;
  __syncthreads();
  if (g == 0 && e < entries) {
    for (int k = 1; k < 16; ++k) a += part[k][threadIdx.x];
    M[(size_t)row * entries + e] = a;
  }
}

// Clears S; 1/q and e/q_c of every q.  On a uniform mesh q_c is the centre of
// the q's group of 4, counted within blocks of 32 (debye_kernel's weights).
__global__ void mesh_kernel(const double *__restrict__ q, unsigned nq, double dq, int uniform,
                            double2 *__restrict__ qe, double *__restrict__ S, size_t ssize) {
  const size_t n = gridDim.x * (size_t)blockDim.x;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < std::max<size_t>(nq, ssize);
       i += n) {
    if (i < ssize) S[i] = 0.0;
    if (i < nq) {
      const double v = q[i];
      double c = v;
      if (uniform) c = fma((double)((i % 32) / 4 * 4) + 1.5, dq, q[i / 32 * 32]);
      qe[i] = make_double2(v == 0.0 ? 0.0 : 1.0 / v, c > 0.0 ? 1e-8 / c : 0.0);
    }
  }
}

// S[row][q] += sum over a chunk's nodes; grid (chunks, q blocks, row groups).
constexpr int kEvalNodes = 64;
template <int RG>
__global__ __launch_bounds__(256) void eval_kernel(const double *__restrict__ M, unsigned nb, int K,
                                                   unsigned cb, double h, unsigned nrows,
                                                   const double *__restrict__ q,
                                                   const double2 *__restrict__ qe, unsigned nq,
                                                   double *__restrict__ S) {
  __shared__ double2 tab[64];
  __shared__ double ct[kMaxMoments * kMaxMoments];  // T_k(t_m) 2/K (k = 0: 1/K)
  __shared__ double4 node[kEvalNodes];              // r/2pi, weight of 1, weight of -e/q_c
  __shared__ double W[kEvalNodes][RG];
  const unsigned b0 = blockIdx.x * cb, nbin = min(cb, nb + 1 - b0);
  const unsigned row0 = blockIdx.z * RG;
  if (threadIdx.x < 64) {
    double s, c;
    sincos_2pi((double)threadIdx.x / 64.0, &s, &c);
    tab[threadIdx.x] = make_double2(s, c);
  }
  for (int i = threadIdx.x; i < K * K; i += 256) {
    const int m = i / K, k = i % K;
    double s, c;
    sincos_2pi((double)((k * (2 * m + 1)) % (4 * K)) / (double)(4 * K), &s, &c);
    ct[i] = (k ? 2.0 * c : 1.0) / K;
  }
  __syncthreads();
  for (unsigned i = threadIdx.x; i < nbin * K; i += 256) {
    const unsigned b = b0 + i / K;
    const int m = i % K;
    const double t = 0.5 * K * ct[m * K + 1];
    const double r = ((b == nb ? 0.0 : (double)b) + 0.5 + 0.5 * t) * h, ir = 1.0 / r;
    node[i] = make_double4(r / kTwoPi, b == nb ? 0.0 : ir,
                           b == nb ? ir : b == 0 ? 0.0 : ir * ir, 0.0);
  }
  for (unsigned i = threadIdx.x; i < nbin * K * RG; i += 256) {
    const unsigned n = i / RG, g = i % RG, row = row0 + g;
    double w = 0.0;
    if (row < nrows) {
      const double *mk = M + ((size_t)row * (nb + 1) + b0 + n / K) * K;
      const double *c = ct + (n % K) * K;
      for (int k = 0; k < K; ++k) w = fma(mk[k], c[k], w);
    }
    W[n][g] = w;
  }
  __syncthreads();
  const unsigned iq = blockIdx.y * 256 + threadIdx.x;
  const double qv = iq < nq ? q[iq] : 0.0;
  const double2 e = iq < nq ? qe[iq] : make_double2(0.0, 0.0);
  double acc[RG];
#pragma unroll
  for (int g = 0; g < RG; ++g) acc[g] = 0.0;
  for (unsigned n = 0; n < nbin * K; ++n) {
    const double4 v = node[n];
    double s, c;
    sincos_2pi_tab(qv * v.x, tab, &s, &c);
    const double f = s * fma(-e.y, v.z, v.y);
#pragma unroll
    for (int g = 0; g < RG; ++g) acc[g] = fma(W[n][g], f, acc[g]);
  }
  if (iq >= nq) return;
#pragma unroll
  for (int g = 0; g < RG; ++g)
    if (row0 + g < nrows && acc[g] != 0.0)
      atomicAdd(&S[(size_t)(row0 + g) * nq + iq], acc[g] * e.x);
}

// ---------------------------------------------------------------- host side
namespace {

struct SegPair {
  uint32_t row, a, b;
};

constexpr int kMoments[] = {6, 8, 10, 12, 14, 18, 24};

// Cycles of the CUs for one call, to choose K and to leave small inputs to
// debye_kernel.  Measured: 143 cycles a wave of 64 pairs for K = 8 on the
// 8,000-atom rock-salt cube (1,560 bins) and 250 for K = 12 on 5,000 atoms
// (290 bins), about 20 a moment; the evaluation's sines at half the issue
// rate; 25 us for the launches and the copy of the tables.
double moments_cycles(double pairs, double rows, double rgroups, unsigned nq, const nodes::Bins &b,
                      double cus) {
  const double per_pair = 20.0 * b.K / 64.0;
  const double node_q = (double)b.entries() * nq * 2.0 * (26.0 * rgroups + 1.5 * rows) / 64.0;
  return pairs * per_pair / cus + node_q / cus + (double)b.entries() * 1.5 + 60000.0;
}
// 3.28 VALU instructions per pair and q at 67% issue, for q in blocks of 1,024
// whether filled or not (340 atoms, 714 q: 85 us; 594 atoms, 1,037 q: 107 us,
// against 50 us through the moments)
double direct_cycles(double pairs, unsigned nq, double cus) {
  return pairs * std::ceil(nq / 1024.0) * 1024.0 * (3.28 / 0.67) / 64.0 / cus + 60000.0;
}

template <int K>
int launch_moments(hipStream_t st, unsigned nruns, size_t lds, const double *xyz, size_t n,
                   const Run *runs, double *slabs, const nodes::Bins &b, int s, unsigned shift) {
  XS_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&moments_kernel<K>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMLds));
  hipLaunchKernelGGL(moments_kernel<K>, dim3(nruns), dim3(kMBlock), lds, st, xyz, xyz + n,
                     xyz + 2 * n, runs, slabs, 1.0 / b.h, b.nb, std::ldexp(1.0, s),
                     std::ldexp(1.0, -s), shift);
  return XS_OK;
}

template <int RG>
void launch_eval(hipStream_t st, dim3 grid, const double *M, const nodes::Bins &b, unsigned cb,
                 unsigned nrows, const double *q, const double2 *qe, unsigned nq, double *S) {
  hipLaunchKernelGGL(eval_kernel<RG>, grid, dim3(256), 0, st, M, b.nb, b.K, cb, b.h, nrows, q, qe,
                     nq, S);
}

}  // namespace

bool plan_moments(const MeshBox &in, const std::vector<uint32_t> &seg_cnt, unsigned n_el,
                  unsigned nblocks, unsigned nq, int cus, MomentPlan *plan) {
  if (!in.finite || !(in.R > 1e-100 && in.R < 1e100) || !(in.Q > 1e-100 && in.Q < 1e100))
    return false;
  const unsigned nparts = nblocks * (nblocks + 1) / 2;
  const double rows = (double)ntypes_of(n_el) * nparts;
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
    if (b.nb > 1000000u || lds_bytes(b.nb, K) > kMLds) continue;
    // each segment pair has at least one slab
    const double slabs = (5.0 * rows + cus) * (double)b.entries() * 8.0;
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

int run_moments(xs_ctx *ctx, const MomentPlan &plan, const double *xyz, size_t n,
                const std::vector<uint32_t> &seg_cnt, unsigned n_el, unsigned nblocks,
                const MeshBox &in, const double *q, unsigned nq, double *S, void *work) {
  const nodes::Bins &b = plan.bins;
  const unsigned nparts = nblocks * (nblocks + 1) / 2;
  const unsigned nrows = ntypes_of(n_el) * nparts;
  std::vector<uint32_t> off(seg_cnt.size() + 1, 0);
  for (size_t s = 0; s < seg_cnt.size(); ++s) off[s + 1] = off[s] + seg_cnt[s];
  // segment pairs by row: (element a, block i) with (element b, block j)
  std::vector<SegPair> sp;
  uint64_t total = 0;
  auto tiles = [&](uint32_t s) { return (uint64_t)(seg_cnt[s] + kMTile - 1) / kMTile; };
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
  unsigned shift = 0;
  while (shift < 3 && (total << shift) < 64ull * ctx->cu_count) ++shift;
  // runs: the shortest longest run for which the segment pairs' runs fill one
  // round of work groups (two runs a segment pair where those are many), at
  // most 2^24 pairs each (the fixed-point sums)
  const double cap = 16777216.0 / (kMTile * kMTile);
  const uint64_t most = std::max<uint64_t>(ctx->cu_count, 2 * sp.size());
  double low = 0.0, per = std::max(1.0, (double)total);
  for (int it = 0; it < 50; ++it) {
    const double mid = 0.5 * (low + per);
    uint64_t nr = 0;
    for (const SegPair &v : sp) nr += (uint64_t)std::ceil((double)pair_tiles(v) / mid);
    (nr <= most ? per : low) = mid;
  }
  per = std::min(per, cap);
  std::vector<Run> runs;
  std::vector<uint32_t> row_run(nrows + 1, 0);
  uint32_t longest = 1;
  for (const SegPair &v : sp) {
    const uint64_t t = pair_tiles(v) << shift;
    if (t) {
      const uint64_t nr = (uint64_t)std::ceil((double)pair_tiles(v) / per);
      for (uint64_t k = 0; k < nr; ++k) {
        const uint64_t f = t * k / nr, e = t * (k + 1) / nr;
        if (e == f) continue;
        runs.push_back(Run{(uint32_t)f, (uint32_t)(e - f), off[v.a], seg_cnt[v.a], off[v.b],
                           seg_cnt[v.b], v.a == v.b ? 1u : 0u, 0u});
        longest = std::max(longest, (uint32_t)(e - f));
      }
    }
    row_run[v.row + 1] = (uint32_t)runs.size();
  }
  for (unsigned r = 0; r < nrows; ++r) row_run[r + 1] = std::max(row_run[r + 1], row_run[r]);
  // |T_k 2^s + ...| <= 2^s per pair: a run's sum stays below 2^62
  const double run_pairs = (double)longest * kMTile * (kMTile >> shift);
  const int s = std::min(48, 62 - (int)std::ceil(std::log2(run_pairs + 1.0)));

  const size_t entries = b.entries();
  char *w = static_cast<char *>(work);
  const size_t rb = runs.size() * sizeof(Run), wb = row_run.size() * 4;
  XS_TRY(ensure_pinned(ctx, align_up(rb, 256) + wb));
  std::memcpy(ctx->pin, runs.data(), rb);
  std::memcpy(static_cast<char *>(ctx->pin) + align_up(rb, 256), row_run.data(), wb);
  Run *runs_d = reinterpret_cast<Run *>(w);
  uint32_t *row_d = reinterpret_cast<uint32_t *>(w + align_up(rb, 256));
  XS_TRY(ensure_matrix(ctx, (runs.size() + nrows) * entries * 8 + (size_t)nq * 16 + 1024));
  double *slabs = static_cast<double *>(ctx->mat);
  double *M = slabs + runs.size() * entries;
  double2 *qe = reinterpret_cast<double2 *>(
      static_cast<char *>(ctx->mat) + align_up((runs.size() + nrows) * entries * 8, 256));
  hipStream_t st = ctx->stream;
  XS_HIP_CHECK(hipMemcpyAsync(runs_d, ctx->pin, align_up(rb, 256) + wb, hipMemcpyHostToDevice, st));
  const size_t ssize = (size_t)nrows * nq;
  hipEvent_t ev;
  XS_TRY(prof_begin(ctx, "debye", &ev));
  hipLaunchKernelGGL(mesh_kernel,
                     dim3((unsigned)std::min<size_t>((std::max<size_t>(ssize, nq) + 255) / 256, 4096)),
                     dim3(256), 0, st, q, nq, in.dq, in.uniform ? 1 : 0, qe, S, ssize);
  if (!runs.empty()) {
    const unsigned nr = (unsigned)runs.size();
    const size_t lds = lds_bytes(b.nb, b.K);
    switch (b.K) {
      case 6: XS_TRY(launch_moments<6>(st, nr, lds, xyz, n, runs_d, slabs, b, s, shift)); break;
      case 8: XS_TRY(launch_moments<8>(st, nr, lds, xyz, n, runs_d, slabs, b, s, shift)); break;
      case 10: XS_TRY(launch_moments<10>(st, nr, lds, xyz, n, runs_d, slabs, b, s, shift)); break;
      case 12: XS_TRY(launch_moments<12>(st, nr, lds, xyz, n, runs_d, slabs, b, s, shift)); break;
      case 14: XS_TRY(launch_moments<14>(st, nr, lds, xyz, n, runs_d, slabs, b, s, shift)); break;
      case 18: XS_TRY(launch_moments<18>(st, nr, lds, xyz, n, runs_d, slabs, b, s, shift)); break;
      default: XS_TRY(launch_moments<24>(st, nr, lds, xyz, n, runs_d, slabs, b, s, shift)); break;
    }
    hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)((entries + 63) / 64), nrows), dim3(1024), 0, st,
                       slabs, row_d, (unsigned)entries, M);
    const unsigned groups = (nrows + 7) / 8, rg = (nrows + groups - 1) / groups;
    const unsigned cb = std::max(1, kEvalNodes / b.K);
    const dim3 grid((b.nb + 1 + cb - 1) / cb, (nq + 255) / 256, (nrows + rg - 1) / rg);
    switch (rg) {
      case 1: launch_eval<1>(st, grid, M, b, cb, nrows, q, qe, nq, S); break;
      case 2: launch_eval<2>(st, grid, M, b, cb, nrows, q, qe, nq, S); break;
      case 3: launch_eval<3>(st, grid, M, b, cb, nrows, q, qe, nq, S); break;
      case 4: launch_eval<4>(st, grid, M, b, cb, nrows, q, qe, nq, S); break;
      case 5: launch_eval<5>(st, grid, M, b, cb, nrows, q, qe, nq, S); break;
      case 6: launch_eval<6>(st, grid, M, b, cb, nrows, q, qe, nq, S); break;
      case 7: launch_eval<7>(st, grid, M, b, cb, nrows, q, qe, nq, S); break;
      default: launch_eval<8>(st, grid, M, b, cb, nrows, q, qe, nq, S); break;
    }
  }
  XS_HIP_CHECK(hipGetLastError());
  return prof_end(ctx, "debye", ev);
}

size_t moments_table_bytes(const std::vector<uint32_t> &seg_cnt, unsigned n_el, unsigned nblocks,
                           int cus) {
  const size_t nparts = (size_t)nblocks * (nblocks + 1) / 2;
  const size_t rows = (size_t)ntypes_of(n_el) * nparts;
  double n = 0.0;
  for (uint32_t c : seg_cnt) n += c;
  const size_t tiles = (size_t)(n / kMTile) + seg_cnt.size();
  const size_t by_cap = (size_t)((double)tiles * (double)tiles / 2 / 4096.0) + 1;
  return align_up((6 * rows + cus + by_cap) * sizeof(Run), 256) + (rows + 1) * 4;
}

}  // namespace debye
}  // namespace xs
