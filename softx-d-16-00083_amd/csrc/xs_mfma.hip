// H3 as a matrix product on the int8 matrix cores (v_mfma_i32_32x32x32_i8).
//
// S[c][q] = sum_k A[q][k] H[c][k],  A[q][k] = sin(q r_k) / (q r_k + 1e-8),
// r_k = (k + 1/2) bin, H = histogram counts (one column c per pair type).
//
// Exact-integer splitting.  A is evaluated in FP64 and split into NA signed
// int8 slices, A = sum_i a_i 2^(-6-7i) + e with |a_0| <= 64, |a_i| <= 64 and
// |e| <= 2^(-7 NA - 0) (the rounding residual of the last slice); counts are
// split exactly into NB 7-bit slices, H = sum_j b_j 2^(7j), b_j in [0, 127].
// Every slice product sum_k a_i b_j is computed exactly by the int8 MFMA in
// int32.  Products with the same d = j - i share the scale 2^(7d-6) and one
// int32 accumulator; accumulators are added into S (FP64) every 32,768 bins,
// before any can overflow (|acc| <= 5 * 64 * 127 * 32768 < 2^31).  All
// NA * NB products are kept: dropping a_4 b_0 would leave an error of
// 2^-28 per count on bins with small counts.  With NA = 5 the result differs
// from the FP64 sum by at most 2^-35 sum_k H[c][k] per entry, against the
// 2^-24-per-term of an FP32 (or split-BF16, FP32 accumulated) product; the
// cancellation of I(q) at its minima amplifies this by up to ~10^4, which
// FP32 accumulation cannot absorb.
//
// Layout.  Slices are stored pre-tiled in the MFMA operand layout: for a
// 32 x 32 (rows x k) tile, lane l holds row l % 32 and k = 16 (l / 32) + j in
// byte j of a 16-byte register group, so a wave loads a tile as one
// contiguous 1 KiB read.  A and B use the same k assignment, which is all the
// product needs.  Accumulator element 4i + jj of lane l is row
// 8i + 4 (l / 32) + jj, column l % 32.
//
// Work groups: 4 waves stacked along q (128 q) x 1 or 2 side by side of NT tiles
// of 32 columns, in equal shares of all k tiles; work groups with consecutive
// shares run on the same XCD (consecutive work-group ids go to different XCDs).
//
// The columns (the histograms of a call, or in pairsum_mfma_batch the pair types of
// many structures) come sorted and grouped by xs_mfma_plan.h; each group has its own
// k range and count slices, one launch covers the groups of one slice count, and the
// columns' results go to their rows of S.  In an ensemble a column's extent is its
// structure's bin count and its slices come from its pair count, so nothing is read
// back; in a call of its own both are read off the counts, while the slices of the
// sine are made.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "xs_internal.h"
#include "xs_sincos.h"

namespace xs {
namespace mm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kNA = kMfmaSlicesA;        // sinc slices
constexpr unsigned kFlush = 1024;  // k tiles (of 32 bins) per int32 accumulation
constexpr double kPi = 3.14159265358979323846;

__global__ __launch_bounds__(256) void clear_u32(uint32_t *__restrict__ p, size_t n) {
  const size_t i = blockIdx.x * (size_t)256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// Every column's counts or-ed together (as many 7-bit slices as the largest) and one
// past its last bin that is not empty.  Grid (columns, parts of the bins).  One atomic
// each per work group: a single word for all columns, an atomic per wave, was 97 us
// for 12.6 M counts, whose 100 MB of loads take 20; this takes 20.
__global__ __launch_bounds__(256) void column_stats(const unsigned long long *__restrict__ hist,
                                                    unsigned nhist,
                                                    unsigned long long *__restrict__ bits,
                                                    uint32_t *__restrict__ last) {
  const unsigned k0 = (unsigned)((unsigned long long)nhist * blockIdx.y / gridDim.y);
  const unsigned k1 = (unsigned)((unsigned long long)nhist * (blockIdx.y + 1) / gridDim.y);
  const unsigned long long *h = hist + (size_t)blockIdx.x * nhist;
  unsigned long long m = 0;
  uint32_t l = 0;
#pragma unroll 4
  for (unsigned k = k0 + threadIdx.x; k < k1; k += 256) {
    const unsigned long long v = h[k];
    m |= v;
    l = v ? k + 1 : l;
  }
  for (int o = 32; o > 0; o >>= 1) {
    m |= (unsigned long long)__shfl_xor(m, o);
    l = max(l, (uint32_t)__shfl_xor(l, o));
  }
  __shared__ unsigned long long pm[4];
  __shared__ uint32_t pl[4];
  if ((threadIdx.x & 63) == 0) {
    pm[threadIdx.x >> 6] = m;
    pl[threadIdx.x >> 6] = l;
  }
  __syncthreads();
  if (threadIdx.x) return;
  l = max(max(pl[0], pl[1]), max(pl[2], pl[3]));
  if (gridDim.y == 1) {  // (nothing to add to, nothing cleared)
    bits[blockIdx.x] = (pm[0] | pm[1]) | (pm[2] | pm[3]);
    last[blockIdx.x] = l;
    return;
  }
  if (!l) return;
  atomicOr(&bits[blockIdx.x], (pm[0] | pm[1]) | (pm[2] | pm[3]));
  atomicMax(&last[blockIdx.x], l);
}

// Slices of the sine table: one thread per (q tile, kSincTiles k tiles, lane), 16
// values a k tile, NA slices of 16 bytes.
// A value v goes to N = rint(2^34 v) by one addition: 2^34 v + 1.5 2^52 + B holds
// N + B in its low bits, B = kSliceBias = 64 (1 + 2^7 + 2^14 + 2^21), so the slices are the 7-bit
// fields of the low word less 64 and, signed, the bits from 28 on.  Four values share
// a reciprocal (1/(abcd), two Newton steps), and the sine is advanced by a rotation
// from bin to bin and over the other half-wave's 16 bins.
// 16,384 bins x 8,192 q: 160 us, of which the 671 MB of stores take 131 (a division
// a value and a rounding, conversion, subtraction and product a slice: 265).
constexpr unsigned kSincTiles = 4;
static_assert(kNA == 5, "bit fields of N");
__global__ __launch_bounds__(256) void slice_sinc(const double *__restrict__ q, unsigned nq,
                                                  unsigned nhist, double bin, unsigned MT, unsigned KT,
                                                  v4i *__restrict__ As) {
  const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  const unsigned KG = (KT + kSincTiles - 1) / kSincTiles;
  if (tid >= (size_t)MT * KG * 64) return;
  const unsigned lane = tid & 63, kg = (tid >> 6) % KG, mt = (unsigned)((tid >> 6) / KG);
  const unsigned row = mt * 32 + (lane & 31), half = 16 * (lane >> 5);
  const double qv = row < nq ? q[row] : 0.0, qb = qv * bin;
  // (of four of which a product is taken: beyond 1e60 the values are 0 either way)
  const double qd = fmin(fmax(qb, -1e60), 1e60);
  double s = 0, c = 1, ds = 0, dc = 1, js = 0, jc = 1;
  if (qv != 0.0) {
    const double turns = qb / (2.0 * kPi);
    sincos_2pi(((double)(kg * kSincTiles * 32 + half) + 0.5) * turns, &s, &c);
    sincos_2pi(turns, &ds, &dc);
    sincos_2pi(16.0 * turns, &js, &jc);
  }
  auto rotate = [&](double bs, double bc) {
    const double sn = fma(s, bc, c * bs);
    c = fma(c, bc, -(s * bs));
    s = sn;
  };
  for (unsigned kt = kg * kSincTiles; kt < min(KT, (kg + 1) * kSincTiles); ++kt) {
    const unsigned k0 = kt * 32 + half;
    unsigned w[kNA][4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      double d[4], v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        d[e] = fma((double)(k0 + 4 * g + e) + 0.5, qd, 1e-8);
        v[e] = s;
        rotate(ds, dc);
      }
      const double ab = d[0] * d[1], cd = d[2] * d[3], p = ab * cd;
      double r = __builtin_amdgcn_rcp(p);
      r = fma(fma(-p, r, 1.0), r, r);
      r = fma(fma(-p, r, 1.0), r, r);
      const double rab = r * cd, rcd = r * ab;
      v[0] *= rab * d[1];
      v[1] *= rab * d[0];
      v[2] *= rcd * d[3];
      v[3] *= rcd * d[2];
      unsigned lo[4], hi[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        constexpr double kBias = 6755399441055744.0 + (double)kSliceBias;
        const bool in = qv != 0.0 && k0 + 4 * g + e < nhist;
        const unsigned long long n =
            (unsigned long long)__double_as_longlong(fma(in ? v[e] : 0.0, 17179869184.0, kBias));
        lo[e] = (unsigned)n;
        hi[e] = (unsigned)(n >> 32);
      }
#pragma unroll
      for (int i = 0; i < kNA; ++i) {
        unsigned f[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          f[e] = i == 0 ? __builtin_amdgcn_alignbit(hi[e], lo[e], 28) & 255u
                        : (lo[e] >> (28 - 7 * i)) & 127u;
        const unsigned b = f[0] | f[1] << 8 | f[2] << 16 | f[3] << 24;
        w[i][g] = i == 0 ? b : ((b | 0x80808080u) - 0x40404040u) ^ 0x80808080u;
      }
    }
#pragma unroll
    for (int i = 0; i < kNA; ++i)
      As[((size_t)i * MT * KT + (size_t)mt * KT + kt) * 64 + lane] =
          (v4i){(int)w[i][0], (int)w[i][1], (int)w[i][2], (int)w[i][3]};
    rotate(js, jc);
  }
}

// The tables of few columns as arguments of a launch, which takes half the time of a copy.
constexpr unsigned kInlineCols = 128, kInlineTiles = 16;
struct InlineTables {
  MfmaCol cols[kInlineCols];
  MfmaTile tiles[kInlineTiles];
};
static_assert(sizeof(InlineTables) <= 3072, "kernel arguments");
__global__ __launch_bounds__(128) void put_tables(InlineTables t, MfmaCol *__restrict__ cols, unsigned ncols,
                                                  MfmaTile *__restrict__ tiles, unsigned ntiles) {
  const unsigned i = threadIdx.x;
  if (i < ncols) cols[i] = t.cols[i];
  if (i < ntiles) tiles[i] = t.tiles[i];
}

static void launch_slice_sinc(xs_ctx *ctx, const double *q, unsigned nq, unsigned nhist, double bin,
                              unsigned MT, unsigned KT, v4i *As) {
  const size_t threads = (size_t)MT * ((KT + kSincTiles - 1) / kSincTiles) * 64;
  hipLaunchKernelGGL(slice_sinc, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, ctx->stream, q,
                     nq, nhist, bin, MT, KT, As);
}

// Counts in slices: one thread per (group, column tile t of the group's NT, k tile
// below kt_max, lane); threads past their group's k range return.  Group g's slices
// go to b_off in the layout [nb][NT][kt][64]; columns past ncols and bins past a
// column's nhist are zero.  S, if given, is cleared.
__global__ void slice_counts(const unsigned long long *__restrict__ hist,
                                   const MfmaCol *__restrict__ cols, unsigned ncols,
                                   const MfmaTile *__restrict__ tiles, unsigned tile0,
                                   unsigned ntiles, unsigned kt_max, int nb, int NT,
                                   v4i *__restrict__ Bs, double *__restrict__ S, size_t ssize) {
  const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (S)
    for (size_t i = tid; i < ssize; i += (size_t)gridDim.x * blockDim.x) S[i] = 0.0;
  const size_t per_t = (size_t)kt_max * 64, per_group = per_t * NT;
  if (tid >= per_group * ntiles) return;
  const unsigned g = (unsigned)(tid / per_group);
  const size_t r = tid % per_group;
  const unsigned t = (unsigned)(r / per_t);
  const unsigned kt = (unsigned)((r % per_t) >> 6);
  const unsigned lane = tid & 63;
  const MfmaTile d = tiles[tile0 + g];
  if (kt >= d.kt) return;
  const unsigned cg = t * 32 + (lane & 31);  // column within the group
  const unsigned k0 = kt * 32 + 16 * (lane >> 5);
  unsigned long long cnt[16];
  MfmaCol c{0ull, 0u, 0u};
  if (cg < d.ncol && d.col0 + cg < ncols) c = cols[d.col0 + cg];
#pragma unroll
  for (int j = 0; j < 16; ++j) cnt[j] = k0 + j < c.nhist ? hist[c.hist_off + k0 + j] : 0ull;
  for (int s = 0; s < nb; ++s) {
    int8_t b[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) b[j] = (int8_t)((cnt[j] >> (7 * s)) & 127ull);
    v4i w;
    __builtin_memcpy(&w, b, 16);
    Bs[d.b_off + ((size_t)(s * NT + t) * d.kt + kt) * 64 + lane] = w;
  }
}

// The same value in every lane, in scalar registers (a 64-bit division leaves it in
// vector registers, of which the products have none to spare).
__device__ __forceinline__ unsigned uniform(unsigned v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ unsigned long long uniform(unsigned long long v) {
  return (unsigned long long)uniform((unsigned)(v >> 32)) << 32 | uniform((unsigned)v);
}

// The product.  A work group is 4 waves stacked along q (4 x 32 q) by WN side by
// side, of NT column tiles each.  Per k tile it needs 4 NA A tiles and NB NT WN B
// tiles, 1 KiB each in the pre-tiled layout, so a global_load_lds_dwordx4 of one
// wave writes exactly one tile (lane l's 16 bytes at 16 l).  The tiles go through
// NS LDS stages: those of k tile kt + NS - 1 are fetched while the products of kt
// run, and the products read their operands from LDS (ds_read_b128 at 16 l, no
// bank conflicts).  Each tile is fetched once per work group, tile b by wave
// b mod (4 WN), which costs one barrier per k tile: before it, each wave waits
// for its own loads of stage kt (vmcnt) and for its own reads of stage
// kt - 1 (lgkmcnt); after it, stage kt is complete in LDS and stage kt - 1,
// which is refilled next with k tile kt + NS - 1, is read by no wave.
// The int32 accumulators go to S (FP64) every kFlush k tiles.  There are as many
// work groups as run at a time, and each takes an equal share of all k tiles: a
// wave owns the output of a group that lies in its share as a whole (the first
// flush stores, later ones add); those that are cut are added to the cleared S.
//
// Measured on the 768-histogram workload (768 x 16,384 bins x 8,192 q):
// operands loaded straight into registers kept the MFMA pipe busy 35% of
// the time, waiting on load latency (two waves per SIMD at 250 VGPRs, no
// registers for a prefetch); per-wave LDS stages one k tile ahead, with
// every wave fetching its own copy of the B tiles (9 KiB per wave per k
// tile), 50%.  Two waves side by side (WN = 2) load 14 KiB instead of 24 for the
// products of four waves.  A work group per group and 128 q left CUs idle 40% of the
// time with two slices (a round and a quarter of work groups of unequal length): 530
// us for the products, 400 to 490 in equal shares.  Particles of 500 to 8,000 atoms leave a
// third of the bins empty past each column's last, and half of the columns take one
// slice: as columns of one k range and slice count the products took 790.
//
// The column tiles come in groups of NT WN with their own k range and slices
// (tiles[tile0 + group]: the count slices at b_off, laid out [NB][NT WN][kt][64]);
// A is laid out with KT, at least the largest k range, and the columns go to the
// rows of S that cols[] names.
template <int NA, int NB, int NT, int WN>
__global__ __launch_bounds__(256 * WN, 2) void pairsum_mfma_lds_kernel(const v4i *__restrict__ As,
                                                                const v4i *__restrict__ Bs,
                                                                unsigned MT, unsigned ngrp, unsigned KT,
                                                                unsigned nq, unsigned ncols,
                                                                double *__restrict__ S,
                                                                const MfmaTile *__restrict__ tiles,
                                                                const MfmaCol *__restrict__ cols,
                                                                unsigned tile0, const double *__restrict__ q,
                                                                double bin) {
  constexpr int DMIN = -(NA - 1);
  constexpr int DMAX = NB - 1;
  constexpr int NG = DMAX - DMIN + 1;
  constexpr int NBT = NB * NT * WN;    // B tiles per k tile
  constexpr int TPS = 4 * NA + NBT;    // tiles per stage
  constexpr int NW = 4 * WN;           // waves
  constexpr int NL = (TPS + NW - 1) / NW;  // of which a wave fetches at most NL
  constexpr int NS = WN == 2 ? 5 : 3;  // stages (one work group a CU, or two)
  // loads per stage that every wave issues at least (without the top slices; some
  // waves issue one or two more: waiting for this count still covers their older stage)
  constexpr int VM = (TPS - 4) / NW;
  constexpr int WAIT = VM * (NS - 2);
  static_assert(WAIT <= 15, "vmcnt field");
  __shared__ v4i stage[NS][TPS][64];
  const unsigned lane = threadIdx.x & 63;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned wm = wave % 4, wn = wave / 4;
  typedef __attribute__((address_space(3))) void lds_t;

  // all waves: own LDS reads done, then the barrier; the empty asm keeps the
  // compiler from moving LDS accesses across it
  auto sync_lds = [&]() {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
  };

  // This work group's share of all k tiles, in the order (128 q, group, k tile).  A
  // group's first k tile in that order follows from where its slices begin.
  constexpr unsigned long long kUnit = (unsigned long long)NB * NT * WN * 64;
  const unsigned long long b0 = tiles[tile0].b_off;
  const unsigned long long K =
      uniform((tiles[tile0 + ngrp - 1].b_off - b0) / kUnit + tiles[tile0 + ngrp - 1].kt);
  const unsigned long long total = K * (MT / 4);
  unsigned share = blockIdx.x;
  if ((gridDim.x & 7u) == 0) share = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  unsigned long long w = uniform(total * share / gridDim.x);
  const unsigned long long wend = uniform(total * (share + 1) / gridDim.x);
  unsigned mg = uniform((unsigned)(w / K)), ng = 0;
  {
    const unsigned long long r = w - mg * K;
    unsigned hi = ngrp - 1;
    while (ng < hi) {
      const unsigned mid = (ng + hi + 1) / 2;
      if ((tiles[tile0 + mid].b_off - b0) / kUnit <= r)
        ng = mid;
      else
        hi = mid - 1;
    }
  }
  ng = uniform(ng);
  unsigned kfirst = uniform((unsigned)(w - mg * K - (tiles[tile0 + ng].b_off - b0) / kUnit));
  while (w < wend) {
    const unsigned mt = mg * 4 + wm;
    // this group's k tiles, B slice stride, B column-tile stride, B base
    const MfmaTile d = tiles[tile0 + ng];
    const unsigned klast = (unsigned)min((unsigned long long)d.kt, kfirst + (wend - w));
    const bool whole = kfirst == 0 && klast == d.kt;
    const size_t sB = (size_t)NT * WN * d.kt * 64, tB = (size_t)d.kt * 64;
    const v4i *bp = Bs + d.b_off;
    const unsigned col0 = d.col0 + wn * NT * 32, colend = min(ncols, d.col0 + d.ncol);

    // Where |q| r > kTopSliceX for all of a q tile, every value's top slice is 0: no
    // products with it from k tile ktop on, no loads from the largest ktop of the work
    // group's q tiles on (kfetch).  (Not asked for 16 k tiles or fewer, whose
    // products take no longer than finding out, 2 us.)
    unsigned ktop = ~0u, kfetch = ~0u;
    if (d.kt > 16) {
      kfetch = 0;
#pragma unroll
      for (unsigned m = 0; m < 4; ++m) {
        const unsigned row = (mg * 4 + m) * 32 + (lane & 31);
        double a = row < nq ? fabs(q[row]) : 0.0;
        a = a > 0.0 ? a : INFINITY;  // (q = 0: a row of zeros; NaN: as it comes)
        for (int o = 16; o > 0; o >>= 1) a = fmin(a, __shfl_xor(a, o, 64));
        const double k = kTopSliceX / (a * bin) * (1.0 / 32.0) + 1.0;
        const unsigned kk = __builtin_amdgcn_readfirstlane(k < 4294967295.0 ? (unsigned)k : ~0u);
        kfetch = max(kfetch, kk);
        if (m == wm) ktop = kk;
      }
    }
    // The tiles of a stage go round the waves: the A tiles (q tile m, slice i > 0) as
    // m (NA - 1) + i - 1, the B tiles (slice j, column tile t) as kB0 + j NT WN + t, and
    // last the top slices, kTop0 + m, which are fetched where a wave needs its own.
    constexpr int kB0 = 4 * (NA - 1), kTop0 = kB0 + NBT;
    const v4i *src[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      const int b = l * NW + (int)wave, c = b - kB0, m = b - kTop0;
      src[l] = c < 0   ? As + ((size_t)(b % (NA - 1) + 1) * MT + mg * 4 + b / (NA - 1)) * KT * 64
               : m < 0 ? bp + (size_t)(c / (NT * WN)) * sB + (size_t)(c % (NT * WN)) * tB
                       : As + ((size_t)mg * 4 + min(m, 3)) * KT * 64;
    }
    auto fetch = [&](unsigned kt, int st) {
      const int tiles_now = kt < kfetch ? TPS : kTop0;
#pragma unroll
      for (int l = 0; l < NL; ++l)
        if (l < VM || l * NW + (int)wave < tiles_now)
          __builtin_amdgcn_global_load_lds((const void *)(src[l] + (size_t)kt * 64 + lane),
                                           (lds_t *)&stage[st][l * NW + wave][0], 16, 0, 0);
    };
    for (unsigned kb = kfirst; kb < klast; kb += kFlush) {
      const unsigned ke = min(klast, kb + kFlush);
      v16i acc[NG][NT];
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[g][t] = v16i{0};
      // no wave still reads a stage of the previous block
      sync_lds();
#pragma unroll
      for (int i = 0; i < NS - 1; ++i)
        if (kb + i < ke) fetch(kb + i, i);
      int st = 0;
      for (unsigned kt = kb; kt < ke; ++kt) {
        if (kt + NS - 2 < ke)
          __builtin_amdgcn_s_waitcnt(0x0f70 | WAIT);  // vmcnt(WAIT): own loads of stage kt landed
        else
          __builtin_amdgcn_s_waitcnt(0x0f70);       // vmcnt(0)
        sync_lds();
        if (kt + NS - 1 < ke) fetch(kt + NS - 1, st == 0 ? NS - 1 : st - 1);
        // the counts first, then the sine's slices one by one, whose products start as
        // they arrive
        v4i a[NA], b[NB][NT];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int t = 0; t < NT; ++t) b[j][t] = stage[st][kB0 + (j * WN + wn) * NT + t][lane];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 1; i < NA; ++i) {
          a[i] = stage[st][wm * (NA - 1) + i - 1][lane];
          __builtin_amdgcn_sched_barrier(0);
        }
        auto multiply = [&](int i) {
#pragma unroll
          for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int t = 0; t < NT; ++t)
              acc[j - i - DMIN][t] =
                  __builtin_amdgcn_mfma_i32_32x32x32_i8(b[j][t], a[i], acc[j - i - DMIN][t], 0, 0, 0);
        };
#pragma unroll
        for (int i = 1; i < NA; ++i) multiply(i);
        if (kt < ktop) {
          a[0] = stage[st][kTop0 + wm][lane];
          multiply(0);
        }
        st = st == NS - 1 ? 0 : st + 1;
      }
      // lane % 32 is a q, so that 32 lanes write 32 consecutive ones of a row.  (Stride
      // and lane are opaque, or addresses would be formed before the loops and kept;
      // the rows' numbers go round by shuffles, as 32 loads a lane would spill.)
      unsigned stride = nq, l = lane;
      __asm__ volatile("" : "+s"(stride), "+v"(l));
      const unsigned row = mt * 32 + (l & 31), half = 4 * (l >> 5);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const unsigned mine = min(col0 + t * 32 + (l & 31), ncols - 1);
        uint32_t type = cols[mine].type;
        __asm__ volatile("" : "+v"(type));
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const unsigned c = 8 * (e >> 2) + (e & 3) + half;
          const size_t srow = (uint32_t)__shfl((int)type, (int)c, 64);
          double v = 0.0;
#pragma unroll
          for (int g = 0; g < NG; ++g) v = fma((double)acc[g][t][e], ldexp(1.0, 7 * (g + DMIN) - 6), v);
          if (row < nq && col0 + t * 32 + c < colend) {
            double *o = S + srow * stride + row;
            if (whole)
              *o = kb == 0 ? v : *o + v;
            else
              atomicAdd(o, v);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    w += klast - kfirst;
    kfirst = klast;
    if (klast == d.kt) {
      kfirst = 0;
      if (++ng == ngrp) {
        ng = 0;
        ++mg;
      }
    }
  }
}

// The products of one slice count's groups.
template <int NT, int WN>
static void launch_gemm(unsigned nb, dim3 grid, hipStream_t st, const v4i *As, const v4i *Bs, unsigned MT,
                        unsigned ngrp, unsigned KT, unsigned nq, unsigned ncols, double *S,
                        const MfmaTile *tiles, const MfmaCol *cols, unsigned tile0, const double *q,
                        double bin) {
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256 * WN), 0, st, As, Bs, MT, ngrp, KT, nq, ncols, S, tiles, cols,
                       tile0, q, bin);
  };
  if constexpr (NT == 2) {  // three count slices with two column tiles would spill
    launch(nb == 1 ? pairsum_mfma_lds_kernel<kNA, 1, NT, WN> : pairsum_mfma_lds_kernel<kNA, 2, NT, WN>);
  } else {
    launch(nb == 3   ? pairsum_mfma_lds_kernel<kNA, 3, NT, WN>
           : nb == 4 ? pairsum_mfma_lds_kernel<kNA, 4, NT, WN>
                     : pairsum_mfma_lds_kernel<kNA, 5, NT, WN>);
  }
}

// Count slices and products of a plan's groups (S is cleared first).
static int products(xs_ctx *ctx, const MfmaBatchPlan &plan, const unsigned long long *hist,
                    const MfmaCol *cols, const MfmaTile *tiles, const v4i *As, v4i *Bs, unsigned KT,
                    double bin, const double *q, unsigned nq, double *S);

}  // namespace mm

static int mm::products(xs_ctx *ctx, const MfmaBatchPlan &plan, const unsigned long long *hist,
                        const MfmaCol *cols, const MfmaTile *tiles, const v4i *As, v4i *Bs, unsigned KT,
                        double bin, const double *q, unsigned nq, double *S) {
  const unsigned MT = (nq + 127) / 128 * 4, ncols = (unsigned)plan.cols.size();
  for (const MfmaLaunch &L : plan.launches) {
    const unsigned NTg = L.nt * L.wn;
    const size_t tb = (size_t)L.ntiles * NTg * plan.kt_max * 64, ssize = (size_t)ncols * nq;
    // (the first one clears S: enough work groups for that too, 100 x 4,000 16 -> 3 us)
    const bool first = &L == &plan.launches[0];
    const size_t groups = std::max((tb + 255) / 256, first ? std::min<size_t>((ssize + 1023) / 1024, 2048) : 0);
    hipLaunchKernelGGL(slice_counts, dim3((unsigned)groups), dim3(256), 0, ctx->stream, hist, cols, ncols,
                       tiles, L.tile0, L.ntiles, plan.kt_max, (int)L.nb, (int)NTg, Bs, first ? S : nullptr,
                       ssize);
  }
  for (const MfmaLaunch &L : plan.launches) {
    // as many work groups as run at a time, of 16 k tiles or one output at least (of
    // short histograms, 9 x 50 bins x 2,000 q, 16 k tiles alone left 2 work groups)
    unsigned long long work = 0;
    for (uint32_t g = 0; g < L.ntiles; ++g) work += plan.tiles[L.tile0 + g].kt;
    work *= MT / 4;
    const unsigned slots = 2 / L.wn * (unsigned)ctx->cu_count;
    const unsigned long long outputs = (unsigned long long)L.ntiles * (MT / 4);
    const dim3 grid((unsigned)std::min<unsigned long long>(slots, std::max(outputs, work / 16)));
    auto gemm = [&](auto launch) {
      launch(L.nb, grid, ctx->stream, As, Bs, MT, L.ntiles, KT, nq, ncols, S, tiles, cols, L.tile0, q, bin);
    };
    if (L.nt == 2 && L.wn == 2)
      gemm(launch_gemm<2, 2>);
    else if (L.nt == 2)
      gemm(launch_gemm<2, 1>);
    else if (L.wn == 2)
      gemm(launch_gemm<1, 2>);
    else
      gemm(launch_gemm<1, 1>);
  }
  XS_HIP_CHECK(hipGetLastError());
  return XS_OK;
}

int pairsum_mfma(xs_ctx *ctx, const unsigned long long *hist, unsigned ncols, unsigned nhist,
                 double bin, const double *q, unsigned nq, double *S, bool host) {
  using namespace mm;
  const unsigned MT = (nq + 127) / 128 * 4;
  const unsigned KT = (nhist + 31) / 32;
  // A small call (not 16 k tiles for every CU): one launch for all slice counts, no waves
  // side by side, which would halve its few work groups (100 x 100 bins x 4,000 q: 59 us
  // side by side and with one launch to clear S, 43 so)
  const bool small = (size_t)(MT / 4) * ((ncols + 127) / 128) * KT < 16 * (size_t)ctx->cu_count;
  const size_t aBytes = (size_t)kNA * MT * KT * 1024;
  XS_TRY(ensure_matrix(ctx, Carver::need({aBytes, (size_t)ncols * 8, (size_t)ncols * 4})));
  XS_TRY(ensure_pinned(ctx, align_up((size_t)ncols * 8, 256) + (size_t)ncols * 4));
  Carver cv(ctx->mat);
  v4i *As = cv.take<v4i>(aBytes / 16);
  unsigned long long *bits = cv.take<unsigned long long>(ncols);
  uint32_t *last = cv.take<uint32_t>(ncols);
  hipEvent_t ev;
  XS_TRY(prof_begin(ctx, "pairsum_slices", &ev));
  // every column's slices and extent, read back while the sine's slices are made
  const unsigned parts = std::min(64u, (nhist + 4095) / 4096);
  const size_t nclear = (size_t)(last + ncols - reinterpret_cast<uint32_t *>(bits));
  if (parts > 1)
    hipLaunchKernelGGL(clear_u32, dim3((unsigned)((nclear + 255) / 256)), dim3(256), 0, ctx->stream,
                       reinterpret_cast<uint32_t *>(bits), nclear);
  hipLaunchKernelGGL(column_stats, dim3(ncols, parts), dim3(256), 0, ctx->stream, hist, nhist, bits, last);
  XS_HIP_CHECK(hipGetLastError());
  // (bits and last in one copy: they lie side by side)
  char *const pin = static_cast<char *>(ctx->pin);
  const size_t last_at = (size_t)(reinterpret_cast<char *>(last) - reinterpret_cast<char *>(bits));
  XS_HIP_CHECK(hipMemcpyAsync(pin, bits, last_at + (size_t)ncols * 4, hipMemcpyDeviceToHost, ctx->stream));
  if (small && host) {
    // (after copies from the host an event's wait takes 6 to 12 us longer than the stream's)
    XS_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    launch_slice_sinc(ctx, q, nq, nhist, bin, MT, KT, As);
    XS_HIP_CHECK(hipGetLastError());
  } else {
    if (!ctx->read_back) XS_HIP_CHECK(hipEventCreateWithFlags(&ctx->read_back, hipEventDisableTiming));
    XS_HIP_CHECK(hipEventRecord(ctx->read_back, ctx->stream));
    launch_slice_sinc(ctx, q, nq, nhist, bin, MT, KT, As);
    XS_HIP_CHECK(hipGetLastError());
    XS_HIP_CHECK(hipEventSynchronize(ctx->read_back));
  }
  std::vector<unsigned long long> off(ncols), bound(ncols);
  std::vector<uint32_t> extent(ncols);
  std::memcpy(bound.data(), pin, (size_t)ncols * 8);
  std::memcpy(extent.data(), pin + last_at, (size_t)ncols * 4);
  for (unsigned c = 0; c < ncols; ++c) off[c] = (unsigned long long)c * nhist;
  if (small) {
    unsigned long long all = 0;
    for (unsigned long long b : bound) all |= b;
    std::fill(bound.begin(), bound.end(), all);
  }
  MfmaBatchPlan plan;
  if (!mfma_batch_plan(off, extent, bound, nq, &plan, !small)) {
    XS_TRY(prof_end(ctx, "pairsum_slices", ev));
    return fail(XS_ERR_RANGE, "xs_hist_pairsum: a bin count exceeds 2^35 (matrix-core path)");
  }
  const size_t colsb = plan.cols.size() * sizeof(MfmaCol), tilesb = plan.tiles.size() * sizeof(MfmaTile);
  XS_TRY(ensure_aux(ctx, Carver::need({colsb, tilesb, plan.b_bytes})));
  XS_TRY(ensure_pinned(ctx, align_up(colsb, 256) + tilesb));
  Carver ca(ctx->aux);
  MfmaCol *cols = ca.take<MfmaCol>(plan.cols.size());
  MfmaTile *tiles = ca.take<MfmaTile>(plan.tiles.size());
  v4i *Bs = ca.take<v4i>(plan.b_bytes / 16);
  if (plan.cols.size() <= kInlineCols && plan.tiles.size() <= kInlineTiles) {
    InlineTables t{};
    std::copy(plan.cols.begin(), plan.cols.end(), t.cols);
    std::copy(plan.tiles.begin(), plan.tiles.end(), t.tiles);
    hipLaunchKernelGGL(put_tables, dim3(1), dim3(128), 0, ctx->stream, t, cols, (unsigned)plan.cols.size(),
                       tiles, (unsigned)plan.tiles.size());
    XS_HIP_CHECK(hipGetLastError());
  } else {
    std::memcpy(ctx->pin, plan.cols.data(), colsb);
    std::memcpy(static_cast<char *>(ctx->pin) + align_up(colsb, 256), plan.tiles.data(), tilesb);
    XS_HIP_CHECK(hipMemcpyAsync(cols, ctx->pin, align_up(colsb, 256) + tilesb, hipMemcpyHostToDevice, ctx->stream));
  }
  XS_TRY(prof_end(ctx, "pairsum_slices", ev));
  XS_TRY(prof_begin(ctx, "pairsum_mfma", &ev));
  XS_TRY(products(ctx, plan, hist, cols, tiles, As, Bs, KT, bin, q, nq, S));
  XS_TRY(prof_end(ctx, "pairsum_mfma", ev));
  return XS_OK;
}

int pairsum_mfma_batch(xs_ctx *ctx, const MfmaBatchPlan &plan, const unsigned long long *hist,
                       const MfmaCol *cols_d, const MfmaTile *tiles_d, void *a_buf, void *b_buf,
                       double bin, const double *q, unsigned nq, double *S, bool prof) {
  using namespace mm;
  if (nq != plan.nq) return fail(XS_ERR_ARG, "pairsum_mfma_batch: plan made for another nq");
  const unsigned MT = (nq + 127) / 128 * 4;
  hipEvent_t ev{};
  if (prof) XS_TRY(prof_begin(ctx, "batch_pairsum", &ev));
  v4i *As = static_cast<v4i *>(a_buf);
  launch_slice_sinc(ctx, q, nq, plan.kt_max * 32, bin, MT, plan.kt_max, As);
  XS_TRY(products(ctx, plan, hist, cols_d, tiles_d, As, static_cast<v4i *>(b_buf), plan.kt_max, bin, q, nq, S));
  if (prof) XS_TRY(prof_end(ctx, "batch_pairsum", ev));
  return XS_OK;
}

}  // namespace xs
