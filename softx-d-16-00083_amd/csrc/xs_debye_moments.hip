// H5/H6 through Chebyshev moments of the pair distances (xs_nodes.h).
//
// The direct Debye sums cost pairs x nq terms; here each pair costs its
// distance and K moments, and the q mesh meets only nb x K nodes per row of S
// (a pair type, or a pair type and block pair).  Four kernels:
//   moments  one work group per run of 64 x 64-atom tile pairs of one segment
//            pair; the moments of all bins live in LDS.  T_0 is a uint32
//            count, T_k (k >= 1) a 64-bit fixed-point sum: T_k 2^48 + 1.5 2^52
//            in one FMA leaves the integer in the low mantissa bits, so the
//            raw bits are added with ds_add_u64 and count x bits(1.5 2^52) is
//            subtracted at the end.  A moment is rounded at 2^-49 per pair
//            whatever the structure's size: the waves meet every kStageJ J atoms,
//            and before a bin could pass 32,767 pairs, where its sums could
//            overflow, the sums go to the run's slab in FP64 and start again.
//            ds_add_u64 on random bins takes 11.4
//            CU cycles a wave, ds_add_u32 6.2, ds_add_f64 21.7 (measured;
//            an odd 8-byte stride between bins, an even one takes 3 times as
//            long): the kernel is bound by these LDS atomics: 143 of the
//            172 CU cycles that 64 pairs take at K = 12 (50,000 atoms); its 90
//            VALU instructions, 57% of the cycles, run beside them.
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

constexpr int kMBlock = 1024;
constexpr double kMagic = 6755399441055744.0;            // 1.5 * 2^52
constexpr unsigned long long kMagicBits = 0x4338000000000000ull;
constexpr unsigned kStageJ = 16;                     // J atoms between two looks at the counts
constexpr unsigned kStagePairs = kMBlock * kStageJ;  // in one bin at most
constexpr unsigned kMaxPairs = 32767;                // |sum of T_k 2^48| < 2^63
static_assert(kStagePairs < kMaxPairs, "a stage must fit");

__device__ __forceinline__ double lane_value(double v, int lane) {
  const unsigned long long u = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)u, lane);
  const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
  return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}

template <int K>
__global__ __launch_bounds__(kMBlock) void moments_kernel(
    const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
    const Run *__restrict__ runs, double *__restrict__ slabs, double inv_h, unsigned nb,
    unsigned sub_shift) {
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
  double *slab = slabs + (size_t)blockIdx.x * ((size_t)nb + 1) * K;
  // The sums so far, added to the slab (the first time: stored) by the whole work
  // group; they start again from zero.
  bool stored = false;
  auto flush = [&]() {
    for (unsigned e = threadIdx.x; e < nb * K; e += kMBlock) {
      const unsigned b = e / K, k = e % K;
      const unsigned long long n = cnt[b];
      double v = (double)n;
      if (k) {
        unsigned long long *p = mom + b * (K - 1) + k - 1;
        v = (double)(long long)(*p - n * kMagicBits) * 0x1p-48;
        *p = 0;
      }
      slab[e] = stored ? slab[e] + v : v;
    }
    stored = true;
    __syncthreads();
    for (unsigned b = threadIdx.x; b < nb; b += kMBlock) cnt[b] = 0;
    __syncthreads();
  };
  __syncthreads();
  for (uint64_t m0 = run.first; m0 < run.first + run.count; m0 += kMBlock / 64) {
    const uint64_t m = m0 + wave;
    const bool item = m < run.first + run.count;  // (else the wave only meets the others)
    const unsigned sub = (unsigned)m & ((1u << sub_shift) - 1);
    const TilePair tp = tile_pair((item ? m : m0) >> sub_shift, TB, run.diag);
    const unsigned ti = __builtin_amdgcn_readfirstlane(tp.ti), tj = __builtin_amdgcn_readfirstlane(tp.tj);
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
    const unsigned jend = item ? min(sub * jr + jr, (run.cntB - tj + TB - 1) / TB) : 0u;
    for (unsigned j0 = sub * jr; j0 < sub * jr + jr; j0 += kStageJ) {
      const unsigned j1 = min(j0 + kStageJ, jend);
      for (unsigned j = j0; j < j1; ++j) {
        const double dx = xi - lane_value(xj, j), dy = yi - lane_value(yj, j),
                     dz = zi - lane_value(zj, j);
        const double s = fma(dx, dx, fma(dy, dy, dz * dz));
        if (j >= jmin && s > 0.0) {
          const double r = sqrt(s);
          const double u = r * inv_h;
          const unsigned b = min((unsigned)u, nb - 1);
          const double t = fma(2.0, __builtin_amdgcn_fract(u), -1.0);
          __hip_atomic_fetch_add(&cnt[b], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          unsigned long long *p = mom + b * (K - 1);
          double tp0 = 1.0, tp1 = t;
          const double t2 = t + t;
#pragma unroll
          for (int k = 1; k < K; ++k) {
            const unsigned long long v = __double_as_longlong(fma(tp1, 0x1p48, kMagic));
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
      __syncthreads();
      bool full = false;
      for (unsigned b = threadIdx.x; b < nb; b += kMBlock) full |= cnt[b] > kMaxPairs - kStagePairs;
      if (__syncthreads_or(full)) flush();
    }
  }
  flush();
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

// e / q_c of q point i.  On a uniform mesh q_c is the centre of the point's group of
// 4, counted within blocks of 32 (debye_kernel's weights).
struct Mesh {
  const double *q;
  unsigned nq;
  double dq;
  int uniform;
};
__device__ __forceinline__ double eps_over_q(const Mesh &m, unsigned i) {
  const double c = m.uniform ? fma((double)((i % 32) / 4 * 4) + 1.5, m.dq, m.q[i / 32 * 32]) : m.q[i];
  return c > 0.0 ? 1e-8 / c : 0.0;
}

// hi + lo += v, without an error in hi + lo (Knuth's two-sum).
__device__ __forceinline__ void add_exact(double &hi, double &lo, double v) {
#pragma clang fp contract(off)
  const double s = hi + v, b = s - hi;
  lo += (hi - (s - b)) + (v - b);
  hi = s;
}

// The same while |hi| >= |v| (Dekker); where hi is smaller, near a zero of the sum, v is
// rounded as it would be anyway.
__device__ __forceinline__ void add_to_larger(double &hi, double &lo, double v) {
#pragma clang fp contract(off)
  const double s = hi + v;
  lo += v - (s - hi);
  hi = s;
}

// part[share][row][q] = q times the sum over a share's nodes, chunk by chunk (every
// gridDim.x-th); grid (shares, q blocks, row groups).
// A node stands for many pairs, so its phase q r is carried beyond FP64 (turn: h / 2 pi
// in two parts): rounded, as a single pair's may be, its error would be the same for
// all of them.  And the nodes run along r, so that the sum grows to many times its
// end value and back at low q: the sums of 8 nodes are added up without rounding.
// 1,500 atoms, q to 20 1/A: 1.2e-16 sqrt(pairs) at high q and 2e-15 max |S| at low q, as
// the sums pair by pair; 2e-15 and 6e-14 with neither.
constexpr int kEvalNodes = 64;
static_assert(kMaxMoments <= kEvalNodes, "a bin a chunk at least");
constexpr unsigned kExactNodes = 4;  // whose sum is rounded
template <int RG>
__global__ __launch_bounds__(256) void eval_kernel(const double *__restrict__ M, unsigned nb, int K,
                                                   unsigned cb, double h, double2 turn, unsigned nrows,
                                                   Mesh mesh, double *__restrict__ part) {
  __shared__ double2 tab[64];
  __shared__ double ct[kMaxMoments * kMaxMoments];  // T_k(t_m) 2/K (k = 0: 1/K)
  __shared__ double4 node[kEvalNodes];              // r/2pi, weight of 1, of -e/q_c; rest of r/2pi
  __shared__ double W[kEvalNodes][RG];
  const unsigned row0 = blockIdx.z * RG, iq = blockIdx.y * 256 + threadIdx.x, nq = mesh.nq;
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
  const double qv = iq < nq ? mesh.q[iq] : 0.0, eq = iq < nq ? eps_over_q(mesh, iq) : 0.0;
  double sum[RG], rest[RG];
#pragma unroll
  for (int g = 0; g < RG; ++g) sum[g] = rest[g] = 0.0;
  for (unsigned b0 = blockIdx.x * cb; b0 <= nb; b0 += gridDim.x * cb) {
    const unsigned nbin = min(cb, nb + 1 - b0), nn = (nbin * K + kExactNodes - 1) / kExactNodes * kExactNodes;
    __syncthreads();
    for (unsigned i = threadIdx.x; i < nn; i += 256) {
      const unsigned b = b0 + i / K;
      const int m = i % K;
      const double t = 0.5 * K * ct[m * K + 1];
      // r / h as x + dx (t to FP64: its bin's share of the distance is small)
      const double c = (b == nb ? 0.0 : (double)b) + 0.5, x = fma(0.5, t, c);
      const double dx = fma(0.5, t, c - x), ir = 1.0 / (x * h), rt = x * turn.x;
      // (beyond the last node: any, of weight 0)
      node[i] = make_double4(rt, b == nb ? 0.0 : ir, b == nb ? ir : b == 0 ? 0.0 : ir * ir,
                             fma(x, turn.x, -rt) + fma(x, turn.y, dx * turn.x));
    }
    for (unsigned i = threadIdx.x; i < nn * RG; i += 256) {
      const unsigned n = i / RG, g = i % RG, row = row0 + g;
      double w = 0.0;
      if (row < nrows && n < nbin * K) {
        const double *mk = M + ((size_t)row * (nb + 1) + b0 + n / K) * K;
        const double *c = ct + (n % K) * K;
        for (int k = 0; k < K; ++k) w = fma(mk[k], c[k], w);
      }
      W[n][g] = w;
    }
    __syncthreads();
    for (unsigned n0 = 0; n0 < nn; n0 += kExactNodes) {
      double acc[RG];
#pragma unroll
      for (int g = 0; g < RG; ++g) acc[g] = 0.0;
#pragma unroll
      for (unsigned n = n0; n < n0 + kExactNodes; ++n) {
        const double4 v = node[n];
        double s, c;
        sincos_turn_tab(fma(qv, v.w, fma(qv, v.x, -rint(qv * v.x))), tab, &s, &c);
        const double f = s * fma(-eq, v.z, v.y);
#pragma unroll
        for (int g = 0; g < RG; ++g) acc[g] = fma(W[n][g], f, acc[g]);
      }
#pragma unroll
      for (int g = 0; g < RG; ++g) add_to_larger(sum[g], rest[g], acc[g]);
    }
  }
  if (iq >= nq) return;
#pragma unroll
  for (int g = 0; g < RG; ++g)
    if (row0 + g < nrows)
      part[((size_t)blockIdx.x * nrows + row0 + g) * nq + iq] = sum[g] + rest[g];
}

// S[row][q] = sum of the shares / q (part may be S itself: one share); 64 q and 16
// threads a q per work group, grid (q blocks, rows).
__global__ __launch_bounds__(1024) void finish_kernel(const double *part, unsigned shares,
                                                      const double *__restrict__ q, unsigned nq,
                                                      double *S) {
  __shared__ double ph[16][64], pl[16][64];
  const unsigned i = threadIdx.x & 63, g = threadIdx.x >> 6, iq = blockIdx.x * 64 + i;
  const size_t at = (size_t)blockIdx.y * nq + iq, stride = (size_t)gridDim.y * nq;
  double hi = 0.0, lo = 0.0;
  if (iq < nq) {
#pragma unroll 4
    for (unsigned x = g; x < shares; x += 16) add_exact(hi, lo, part[x * stride + at]);
  }
  ph[g][i] = hi;
  pl[g][i] = lo;
  __syncthreads();
  if (g || iq >= nq) return;
  for (unsigned k = 1; k < 16; ++k) {
    add_exact(hi, lo, ph[k][i]);
    lo += pl[k][i];
  }
  const double qv = q[iq];
  S[at] = qv == 0.0 ? 0.0 : (hi + lo) / qv;
}

// ---------------------------------------------------------------- host side
namespace {

template <int K>
int launch_moments(hipStream_t st, unsigned nruns, size_t lds, const double *xyz, size_t n,
                   const Run *runs, double *slabs, const nodes::Bins &b, unsigned shift) {
  XS_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&moments_kernel<K>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMLds));
  hipLaunchKernelGGL(moments_kernel<K>, dim3(nruns), dim3(kMBlock), lds, st, xyz, xyz + n,
                     xyz + 2 * n, runs, slabs, b.inv_h, b.nb, shift);
  return XS_OK;
}

template <int RG>
void launch_eval(hipStream_t st, dim3 grid, const double *M, const nodes::Bins &b, unsigned cb,
                 unsigned nrows, const Mesh &mesh, double *part) {
  const long double h = b.h(), turn = h / 6.283185307179586476925286766559L;
  const double hi = (double)turn;
  hipLaunchKernelGGL(eval_kernel<RG>, grid, dim3(256), 0, st, M, b.nb, b.K, cb, (double)h,
                     make_double2(hi, (double)(turn - hi)), nrows, mesh, part);
}

}  // namespace

int run_moments(xs_ctx *ctx, const MomentPlan &plan, const double *xyz, size_t n,
                const std::vector<uint32_t> &seg_cnt, unsigned n_el, unsigned nblocks,
                const MeshBox &in, const double *q, unsigned nq, double *S, void *work) {
  const nodes::Bins &b = plan.bins;
  const unsigned nparts = nblocks * (nblocks + 1) / 2;
  const unsigned nrows = ntypes_of(n_el) * nparts;
  const RunTables T = plan_runs(seg_cnt, n_el, nblocks, ctx->cu_count);
  const std::vector<Run> &runs = T.runs;
  const std::vector<uint32_t> &row_run = T.row_run;
  const unsigned shift = T.shift;
  const size_t entries = b.entries();
  char *w = static_cast<char *>(work);
  const size_t rb = runs.size() * sizeof(Run), wb = row_run.size() * 4;
  XS_TRY(ensure_pinned(ctx, align_up(rb, 256) + wb));
  std::memcpy(ctx->pin, runs.data(), rb);
  std::memcpy(static_cast<char *>(ctx->pin) + align_up(rb, 256), row_run.data(), wb);
  Run *runs_d = reinterpret_cast<Run *>(w);
  uint32_t *row_d = reinterpret_cast<uint32_t *>(w + align_up(rb, 256));
  // the evaluation: chunks of cb bins (the near pairs' among them), up to 8 rows at once,
  // as many shares of the chunks as give eight work groups a CU
  const size_t ssize = (size_t)nrows * nq;
  const unsigned groups = (nrows + 7) / 8, rg = (nrows + groups - 1) / groups;
  const unsigned cb = std::max(1, kEvalNodes / b.K), chunks = (b.nb + 1 + cb - 1) / cb;
  const size_t eval_groups = (size_t)((nq + 255) / 256) * ((nrows + rg - 1) / rg);
  const unsigned shares =
      runs.empty() ? 0 : (unsigned)std::min<size_t>(chunks, std::max<size_t>(1, 8 * ctx->cu_count / eval_groups));
  XS_TRY(ensure_matrix(ctx, Carver::need({runs.size() * entries * 8, nrows * entries * 8,
                                          shares > 1 ? shares * ssize * 8 : 0})));
  Carver cv(ctx->mat);
  double *slabs = cv.take<double>(runs.size() * entries), *M = cv.take<double>(nrows * entries);
  double *part = shares > 1 ? cv.take<double>(shares * ssize) : S;
  hipStream_t st = ctx->stream;
  XS_HIP_CHECK(hipMemcpyAsync(runs_d, ctx->pin, align_up(rb, 256) + wb, hipMemcpyHostToDevice, st));
  hipEvent_t ev;
  XS_TRY(prof_begin(ctx, "debye", &ev));
  if (!runs.empty()) {
    const unsigned nr = (unsigned)runs.size();
    const size_t lds = moments_lds_bytes(b.nb, b.K);
    switch (b.K) {
      case 8: XS_TRY(launch_moments<8>(st, nr, lds, xyz, n, runs_d, slabs, b, shift)); break;
      case 10: XS_TRY(launch_moments<10>(st, nr, lds, xyz, n, runs_d, slabs, b, shift)); break;
      case 12: XS_TRY(launch_moments<12>(st, nr, lds, xyz, n, runs_d, slabs, b, shift)); break;
      case 14: XS_TRY(launch_moments<14>(st, nr, lds, xyz, n, runs_d, slabs, b, shift)); break;
      case 18: XS_TRY(launch_moments<18>(st, nr, lds, xyz, n, runs_d, slabs, b, shift)); break;
      case 24: XS_TRY(launch_moments<24>(st, nr, lds, xyz, n, runs_d, slabs, b, shift)); break;
      default: XS_TRY(launch_moments<32>(st, nr, lds, xyz, n, runs_d, slabs, b, shift)); break;
    }
    hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)((entries + 63) / 64), nrows), dim3(1024), 0, st,
                       slabs, row_d, (unsigned)entries, M);
    const dim3 grid(shares, (nq + 255) / 256, (nrows + rg - 1) / rg);
    const Mesh mesh{q, nq, in.dq, in.uniform ? 1 : 0};
    switch (rg) {
      case 1: launch_eval<1>(st, grid, M, b, cb, nrows, mesh, part); break;
      case 2: launch_eval<2>(st, grid, M, b, cb, nrows, mesh, part); break;
      case 3: launch_eval<3>(st, grid, M, b, cb, nrows, mesh, part); break;
      case 4: launch_eval<4>(st, grid, M, b, cb, nrows, mesh, part); break;
      case 5: launch_eval<5>(st, grid, M, b, cb, nrows, mesh, part); break;
      case 6: launch_eval<6>(st, grid, M, b, cb, nrows, mesh, part); break;
      case 7: launch_eval<7>(st, grid, M, b, cb, nrows, mesh, part); break;
      default: launch_eval<8>(st, grid, M, b, cb, nrows, mesh, part); break;
    }
  }
  hipLaunchKernelGGL(finish_kernel, dim3((nq + 63) / 64, nrows), dim3(1024), 0, st, part, shares, q, nq, S);
  XS_HIP_CHECK(hipGetLastError());
  return prof_end(ctx, "debye", ev);
}

}  // namespace debye
}  // namespace xs
