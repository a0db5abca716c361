// Atoms into equal-count tiles on the device: slabs along x, columns along y in each,
// runs along z in each column.
//
// What the histogram kernels need is tiles of equal counts, compact in space; the
// order of atoms within a tile, or of atoms a thousandth of the extent apart, is free.
// So nothing is sorted: an atom counts itself into a bucket of its coordinate (the
// atomic's old value is its place in the bucket), the buckets of a part are summed up,
// and bucket + place is the atom's rank, which gives its slab; then the same within
// the slab for its column, and within the column for its final place.  A part of n
// atoms has n / 4 buckets, 32 to 4,096.
//
// Bound by launches (eight, about 3 us each) and the latency of the atomics.  110,592
// atoms, FP64 (two elements): 47 us; the radix and merge sorts of three 64-bit
// and two 32-bit keys per element took 480 in 110 launches.  Few atoms go through one
// work group in one launch (small).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "xs_order.h"

namespace xs {
namespace order {

constexpr int kThreads = 256;

static uint32_t buckets_for(uint32_t n) {
  uint32_t b = 32;
  while (b < 4096 && b * 8 <= n) b *= 2;
  return b;
}

void Tables::add(uint32_t start, uint32_t n, uint32_t gx, uint32_t gy, const double box[6]) {
  Seg s{};
  s.start = start;
  s.n = n;
  s.gx = gx;
  s.slab0 = (uint32_t)slabs.size();
  s.count0 = (uint32_t)counters;
  s.nb = buckets_for(n);
  counters += s.nb;
  for (int a = 0; a < 3; ++a) {
    const double ext = box[3 + a] - box[a], inv = 1.0 / ext;
    s.lo[a] = box[a];
    s.scale[a] = ext > 0.0 && std::isfinite(inv) ? inv : 0.0;
  }
  for (uint64_t i = 0; i < gx; ++i) {
    const uint32_t a0 = (uint32_t)(i * n / gx), a1 = (uint32_t)((i + 1) * n / gx);
    Slab l{};
    l.start = start + a0;
    l.n = a1 - a0;
    l.gy = gy;
    l.col0 = ncols;
    l.seg = (uint32_t)segs.size();
    l.count0 = (uint32_t)counters;
    l.nb = buckets_for(l.n);
    counters += l.nb;
    l.zcount0 = (uint32_t)counters;
    l.znb = buckets_for(l.n / gy);
    counters += (size_t)l.znb * gy;
    ncols += gy;
    slabs.push_back(l);
  }
  segs.push_back(s);
  natoms += n;
}

void Tables::write_tables(char *dst) const {
  std::memcpy(dst, segs.data(), segs.size() * sizeof(Seg));
  std::memcpy(dst + align_up(segs.size() * sizeof(Seg), 256), slabs.data(), slabs.size() * sizeof(Slab));
}

size_t Tables::scratch_bytes() const {
  return Carver::need({counters * 4, natoms * 4, natoms * 4, natoms * 4});
}

// Part of rank r when n ranks are split into g equal-count parts, part s
// starting at floor(s n / g).
__device__ inline uint32_t equal_part(uint64_t r, uint64_t n, uint64_t g) {
  uint64_t s = r * g / n;
  while (s + 1 < g && (s + 1) * n / g <= r) ++s;
  while (s > 0 && s * n / g > r) --s;
  return (uint32_t)s;
}

__device__ __forceinline__ uint32_t bucket(double v, double lo, double scale, uint32_t nb) {
  const double f = (v - lo) * scale * (double)nb;
  return f >= 0.0 ? (uint32_t)fmin(f, (double)(nb - 1)) : 0u;
}

// The atom's place in its counter.  Lanes that share the first lane's counter (a
// lattice's plane) take theirs with one atomic.
__device__ __forceinline__ uint32_t take_place(uint32_t *__restrict__ count, uint32_t k, bool in) {
  const unsigned lane = threadIdx.x & 63;
  uint32_t place = 0;
  for (int round = 0; round < 3; ++round) {
    const unsigned long long left = __ballot(in);
    if (!left) return place;
    const int first = __ffsll(left) - 1;
    const uint32_t kf = __shfl(k, first, 64);
    const unsigned long long same = __ballot(in && k == kf);
    if (__popcll(same) < 12) break;
    uint32_t base = 0;
    if ((int)lane == first) base = atomicAdd(&count[kf], (uint32_t)__popcll(same));
    base = __shfl(base, first, 64);
    if (in && k == kf) {
      place = base + (uint32_t)__popcll(same & ((1ull << lane) - 1));
      in = false;
    }
  }
  if (in) place = atomicAdd(&count[k], 1u);
  return place;
}

__global__ __launch_bounds__(kThreads) void clear(uint32_t *__restrict__ p, size_t n) {
  const size_t i = blockIdx.x * (size_t)kThreads + threadIdx.x;
  if (i < n) p[i] = 0u;
}

struct Work {
  const Seg *segs;
  const Slab *slabs;
  unsigned nseg, nslab;
  uint32_t *count, *key, *place, *slab;  // key: the atom's counter
  uint32_t natoms;
};

__device__ __forceinline__ unsigned seg_of(const Work &W, uint32_t a) {
  unsigned lo = 0, hi = W.nseg - 1;
  while (lo < hi) {  // the last segment that starts at or before a (empty ones share a start)
    const unsigned mid = (lo + hi + 1) / 2;
    if (W.segs[mid].start <= a)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

template <class S>
__global__ __launch_bounds__(kThreads) void count_x(Work W, const S *__restrict__ x) {
  const uint32_t a = blockIdx.x * kThreads + threadIdx.x;
  const bool in = a < W.natoms;
  uint32_t k = 0;
  if (in) {
    const Seg s = W.segs[seg_of(W, a)];
    k = s.count0 + bucket((double)x[a], s.lo[0], s.scale[0], s.nb);
    W.key[a] = k;
  }
  const uint32_t p = take_place(W.count, k, in);
  if (in) W.place[a] = p;
}

template <class S>
__global__ __launch_bounds__(kThreads) void count_y(Work W, const S *__restrict__ y) {
  const uint32_t a = blockIdx.x * kThreads + threadIdx.x;
  const bool in = a < W.natoms;
  uint32_t k = 0;
  if (in) {
    const Seg s = W.segs[seg_of(W, a)];
    const uint32_t rank = W.count[W.key[a]] + W.place[a];
    const uint32_t i = s.slab0 + equal_part(rank - s.start, s.n, s.gx);
    const Slab l = W.slabs[i];
    k = l.count0 + bucket((double)y[a], s.lo[1], s.scale[1], l.nb);
    W.key[a] = k;
    W.slab[a] = i;
  }
  const uint32_t p = take_place(W.count, k, in);
  if (in) W.place[a] = p;
}

template <class S>
__global__ __launch_bounds__(kThreads) void count_z(Work W, const S *__restrict__ z) {
  const uint32_t a = blockIdx.x * kThreads + threadIdx.x;
  const bool in = a < W.natoms;
  uint32_t k = 0;
  if (in) {
    const Slab l = W.slabs[W.slab[a]];
    const uint32_t rank = W.count[W.key[a]] + W.place[a];
    const uint32_t c = equal_part(rank - l.start, l.n, l.gy);
    k = l.zcount0 + c * l.znb + bucket((double)z[a], W.segs[l.seg].lo[2], W.segs[l.seg].scale[2], l.znb);
    W.key[a] = k;
  }
  const uint32_t p = take_place(W.count, k, in);
  if (in) W.place[a] = p;
}

// Counters c[0, nb) become the first rank of each bucket, the part's ranks beginning
// at `start`.  One work group.
__device__ void sum_buckets(uint32_t *__restrict__ c, uint32_t nb, uint32_t start) {
  __shared__ uint32_t part[kThreads / 64];
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t carry = start;
  for (uint32_t base = 0; base < nb; base += 4 * kThreads) {
    const uint32_t i = base + 4 * threadIdx.x;
    uint32_t v[4], sum = 0;
    for (int j = 0; j < 4; ++j) {
      const uint32_t n = i + j < nb ? c[i + j] : 0u;
      v[j] = sum;
      sum += n;
    }
    uint32_t incl = sum;
    for (int d = 1; d < 64; d *= 2) {
      const uint32_t o = __shfl_up(incl, d, 64);
      if ((int)lane >= d) incl += o;
    }
    __syncthreads();
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    uint32_t before = carry + incl - sum;
    for (unsigned w = 0; w < kThreads / 64; ++w) {
      if (w < wave) before += part[w];
      carry += part[w];
    }
    for (int j = 0; j < 4; ++j)
      if (i + j < nb) c[i + j] = before + v[j];
  }
}

__global__ __launch_bounds__(kThreads) void sum_x(Work W) {
  const Seg s = W.segs[blockIdx.x];
  sum_buckets(W.count + s.count0, s.nb, s.start);
}

__global__ __launch_bounds__(kThreads) void sum_y(Work W) {
  const Slab l = W.slabs[blockIdx.x];
  sum_buckets(W.count + l.count0, l.nb, l.start);
}

__global__ __launch_bounds__(kThreads) void sum_z(Work W, uint32_t ncols) {
  for (uint32_t col = blockIdx.x; col < ncols; col += gridDim.x) {
    unsigned lo = 0, hi = W.nslab - 1;
    while (lo < hi) {
      const unsigned mid = (lo + hi + 1) / 2;
      if (W.slabs[mid].col0 <= col)
        lo = mid;
      else
        hi = mid - 1;
    }
    const Slab l = W.slabs[lo];
    const uint64_t c = col - l.col0;
    sum_buckets(W.count + l.zcount0 + c * l.znb, l.znb, l.start + (uint32_t)(c * l.n / l.gy));
  }
}

template <class S, class T>
__global__ __launch_bounds__(kThreads) void put(Work W, const S *__restrict__ x, const S *__restrict__ y,
                                                const S *__restrict__ z, T *__restrict__ sx,
                                                T *__restrict__ sy, T *__restrict__ sz) {
  const uint32_t a = blockIdx.x * kThreads + threadIdx.x;
  if (a >= W.natoms) return;
  const uint32_t p = W.count[W.key[a]] + W.place[a];
  sx[p] = (T)x[a];
  sy[p] = (T)y[a];
  sz[p] = (T)z[a];
}

// The same by one work group, for up to kSmallAtoms atoms and kSmallCounters counters:
// counters in LDS, an atom's coordinates, counter and place in registers.  Parts follow
// one another in the counters as their atoms do in the ranks, so one sum over all
// counters of an axis gives every atom its rank.  Bound by latency (tables, LDS atomics,
// 15 barriers): 2,000 atoms 14 us, where the eight launches take 27 and their gaps.
// Whole FP64 histograms of 500, 2,000 and 3,000 atoms 134, 149 and 140 -> 118, 138 and 133 us
// (with one launch less each for records and clearing); at 4,096 atoms both ways take 143.5.
constexpr int kSmallThreads = 1024, kSmallPer = 4;
constexpr uint32_t kSmallAtoms = kSmallThreads * kSmallPer, kSmallCounters = 8192;

template <class S, class T>
__global__ __launch_bounds__(kSmallThreads) void small(Work W, const S *__restrict__ x,
                                                       const S *__restrict__ y, const S *__restrict__ z,
                                                       T *__restrict__ sx, T *__restrict__ sy,
                                                       T *__restrict__ sz) {
  __shared__ uint32_t count[kSmallCounters], part[kSmallThreads / 64];
  constexpr uint32_t kOwn = kSmallCounters / kSmallThreads;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  S v[3][kSmallPer] = {};
  uint32_t seg[kSmallPer] = {}, slab[kSmallPer] = {}, rank[kSmallPer] = {}, key[kSmallPer] = {};
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    const uint32_t a = tid + j * kSmallThreads;
    if (a < W.natoms) {
      v[0][j] = x[a];
      v[1][j] = y[a];
      v[2][j] = z[a];
      seg[j] = seg_of(W, a);
    }
  }
#pragma unroll
  for (int axis = 0; axis < 3; ++axis) {
    for (uint32_t i = tid; i < kSmallCounters; i += kSmallThreads) count[i] = 0u;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSmallPer; ++j) {
      const bool in = tid + j * kSmallThreads < W.natoms;
      if (in) {
        const Seg s = W.segs[seg[j]];
        if (axis == 0) {
          key[j] = s.count0 + bucket((double)v[0][j], s.lo[0], s.scale[0], s.nb);
        } else if (axis == 1) {
          slab[j] = s.slab0 + equal_part(rank[j] - s.start, s.n, s.gx);
          const Slab l = W.slabs[slab[j]];
          key[j] = l.count0 + bucket((double)v[1][j], s.lo[1], s.scale[1], l.nb);
        } else {
          const Slab l = W.slabs[slab[j]];
          const uint32_t c = equal_part(rank[j] - l.start, l.n, l.gy);
          key[j] = l.zcount0 + c * l.znb + bucket((double)v[2][j], s.lo[2], s.scale[2], l.znb);
        }
      }
      rank[j] = take_place(count, key[j], in);
    }
    __syncthreads();
    uint32_t before[kOwn], sum = 0;
    for (uint32_t i = 0; i < kOwn; ++i) {
      before[i] = sum;
      sum += count[kOwn * tid + i];
    }
    uint32_t incl = sum;
    for (int d = 1; d < 64; d *= 2) {
      const uint32_t o = __shfl_up(incl, d, 64);
      if ((int)lane >= d) incl += o;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    uint32_t first = incl - sum;
    for (uint32_t w = 0; w < wave; ++w) first += part[w];
    for (uint32_t i = 0; i < kOwn; ++i) count[kOwn * tid + i] = first + before[i];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSmallPer; ++j)
      if (tid + j * kSmallThreads < W.natoms) rank[j] += count[key[j]];
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j)
    if (tid + j * kSmallThreads < W.natoms) {
      sx[rank[j]] = (T)v[0][j];
      sy[rank[j]] = (T)v[1][j];
      sz[rank[j]] = (T)v[2][j];
    }
}

template <class S, class T>
int run(xs_ctx *ctx, const Tables &t, const char *tables, char *scratch, const S *x, const S *y,
        const S *z, T *sx, T *sy, T *sz) {
  if (!t.natoms) return XS_OK;
  if (t.counters > 0xffffffffull) return fail(XS_ERR_RANGE, "histogram: too many atoms over too many bins");
  Carver cv(scratch);
  Work W{};
  W.segs = reinterpret_cast<const Seg *>(tables);
  W.slabs = reinterpret_cast<const Slab *>(tables + align_up(t.segs.size() * sizeof(Seg), 256));
  W.nseg = (unsigned)t.segs.size();
  W.nslab = (unsigned)t.slabs.size();
  W.count = cv.take<uint32_t>(t.counters);
  W.key = cv.take<uint32_t>(t.natoms);
  W.place = cv.take<uint32_t>(t.natoms);
  W.slab = cv.take<uint32_t>(t.natoms);
  W.natoms = (uint32_t)t.natoms;
  const hipStream_t st = ctx->stream;
  if (t.natoms <= kSmallAtoms && t.counters <= kSmallCounters) {
    hipLaunchKernelGGL((small<S, T>), dim3(1), dim3(kSmallThreads), 0, st, W, x, y, z, sx, sy, sz);
    XS_HIP_CHECK(hipGetLastError());
    return XS_OK;
  }
  const dim3 block(kThreads), atoms((unsigned)((t.natoms + kThreads - 1) / kThreads));
  hipLaunchKernelGGL(clear, dim3((unsigned)((t.counters + kThreads - 1) / kThreads)), block, 0, st, W.count,
                     t.counters);
  hipLaunchKernelGGL((count_x<S>), atoms, block, 0, st, W, x);
  hipLaunchKernelGGL(sum_x, dim3(W.nseg), block, 0, st, W);
  hipLaunchKernelGGL((count_y<S>), atoms, block, 0, st, W, y);
  hipLaunchKernelGGL(sum_y, dim3(W.nslab), block, 0, st, W);
  hipLaunchKernelGGL((count_z<S>), atoms, block, 0, st, W, z);
  hipLaunchKernelGGL(sum_z, dim3(std::min(t.ncols, 1u << 20)), block, 0, st, W, t.ncols);
  hipLaunchKernelGGL((put<S, T>), atoms, block, 0, st, W, x, y, z, sx, sy, sz);
  XS_HIP_CHECK(hipGetLastError());
  return XS_OK;
}

template int run<double, double>(xs_ctx *, const Tables &, const char *, char *, const double *,
                                 const double *, const double *, double *, double *, double *);
template int run<double, float>(xs_ctx *, const Tables &, const char *, char *, const double *,
                                const double *, const double *, float *, float *, float *);
template int run<float, float>(xs_ctx *, const Tables &, const char *, char *, const float *,
                               const float *, const float *, float *, float *, float *);

}  // namespace order
}  // namespace xs
