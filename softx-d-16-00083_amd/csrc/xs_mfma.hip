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
// of 32 columns; tiles are ordered so that the work groups that share a q block
// run on the same XCD (consecutive work-group ids go to different XCDs).  Few work
// groups, or a last round of them half empty, share out the k range.
//
// Ensembles (pairsum_mfma_batch): the columns are the pair types of many
// structures, each with its own bin count.  They come sorted and grouped by
// xs_mfma_plan.h; each group of NT column tiles has its own k range and
// count slices, one launch covers the groups of one slice count, and the
// columns' results go to their pair types' rows of S.  The slice count of a
// type comes from its pair count, so nothing is read back.
#include <algorithm>
#include <cmath>

#include "xs_internal.h"
#include "xs_sincos.h"

namespace xs {
namespace mm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kNA = kMfmaSlicesA;        // sinc slices
constexpr int kMaxNB = kMfmaMaxSlicesB;  // count slices (counts < 2^35)
constexpr unsigned kFlush = 1024;  // k tiles (of 32 bins) per int32 accumulation
constexpr double kPi = 3.14159265358979323846;

// All counts or-ed together: as many 7-bit slices as the largest.  A work group adds
// its word only where that brings a new bit (an atomic per wave, 8,192 on one address,
// was 97 us for 12.6 M counts, whose 100 MB of loads take 20; now 21).
__global__ __launch_bounds__(256) void or_u64(const unsigned long long *__restrict__ h, size_t n,
                                              unsigned long long *__restrict__ out) {
  unsigned long long m = 0;
  const size_t step = (size_t)gridDim.x * blockDim.x;
  size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  for (; i + 3 * step < n; i += 4 * step)
    m |= (h[i] | h[i + step]) | (h[i + 2 * step] | h[i + 3 * step]);
  for (; i < n; i += step) m |= h[i];
  for (int o = 32; o > 0; o >>= 1) m |= (unsigned long long)__shfl_xor(m, o);
  __shared__ unsigned long long part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x) return;
  m = (part[0] | part[1]) | (part[2] | part[3]);
  if (m & ~__hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(out, m);
}

__global__ void zero_u64(unsigned long long *p) { *p = 0ull; }

// Slices of the sine table: one thread per (q tile, kSincTiles k tiles, lane), 16
// values a k tile, NA slices of 16 bytes.
// A value v goes to N = rint(2^34 v) by one addition: 2^34 v + 1.5 2^52 + B holds
// N + B in its low bits, B = 64 (1 + 2^7 + 2^14 + 2^21), so the slices are the 7-bit
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
        d[e] = fma((double)(k0 + 4 * g + e) + 0.5, qb, 1e-8);
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
        constexpr double kBias = 6755399441055744.0 + 64.0 * (1 + 128 + 16384 + 2097152);
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

static void launch_slice_sinc(xs_ctx *ctx, const double *q, unsigned nq, unsigned nhist, double bin,
                              unsigned MT, unsigned KT, v4i *As) {
  const size_t threads = (size_t)MT * ((KT + kSincTiles - 1) / kSincTiles) * 64;
  hipLaunchKernelGGL(slice_sinc, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, ctx->stream, q,
                     nq, nhist, bin, MT, KT, As);
}

// One thread per (column tile, k tile, lane): 16 counts, NB 7-bit slices.  S, if
// given, is cleared.
__global__ void slice_counts(const unsigned long long *__restrict__ hist, unsigned ncols,
                             unsigned nhist, unsigned NTn, unsigned KT, int nb,
                             v4i *__restrict__ Bs, double *__restrict__ S, size_t ssize) {
  const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (S)
    for (size_t i = tid; i < ssize; i += (size_t)gridDim.x * blockDim.x) S[i] = 0.0;
  const size_t total = (size_t)NTn * KT * 64;
  if (tid >= total) return;
  const unsigned lane = tid & 63;
  const size_t tile = tid >> 6;
  const unsigned kt = tile % KT;
  const unsigned nt = tile / KT;
  const unsigned col = nt * 32 + (lane & 31);
  const unsigned k0 = kt * 32 + 16 * (lane >> 5);
  unsigned long long cnt[16];
#pragma unroll
  for (int j = 0; j < 16; ++j)
    cnt[j] = (col < ncols && k0 + j < nhist) ? hist[(size_t)col * nhist + k0 + j] : 0ull;
  for (int s = 0; s < nb; ++s) {
    int8_t b[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) b[j] = (int8_t)((cnt[j] >> (7 * s)) & 127ull);
    v4i w;
    __builtin_memcpy(&w, b, 16);
    Bs[(size_t)s * total + tid] = w;
  }
}

// Counts of an ensemble's pair types: one thread per (group, column tile t
// of the group, k tile below kt_max, lane); threads past their group's k
// range return.  Group g's slices go to b_off in the layout [nb][NT][kt][64];
// columns past ncols and bins past a column's nhist are zero.
__global__ void slice_counts_batch(const unsigned long long *__restrict__ hist,
                                   const MfmaCol *__restrict__ cols, unsigned ncols,
                                   const MfmaTile *__restrict__ tiles, unsigned tile0,
                                   unsigned ntiles, unsigned kt_max, int nb, int NT,
                                   v4i *__restrict__ Bs) {
  const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
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

// The product.  A work group is 4 waves stacked along q (4 x 32 q) by WN side by
// side, of NT column tiles each.  Per k tile it needs 4 NA A tiles and NB NT WN B
// tiles, 1 KiB each in the pre-tiled layout, so a global_load_lds_dwordx4 of one
// wave writes exactly one tile (lane l's 16 bytes at 16 l).  The tiles go through
// three LDS stages: those of k tile kt + 2 are fetched while the products of kt
// run, and the products read their operands from LDS (ds_read_b128 at 16 l, no
// bank conflicts).  Each tile is fetched once per work group, tile b by wave
// b mod (4 WN), which costs one barrier per k tile: before it, each wave waits
// for its own loads of stage kt (vmcnt) and for its own reads of stage
// kt - 1 (lgkmcnt); after it, stage kt is complete in LDS and stage kt - 1,
// which is refilled next with k tile kt + 2, is read by no wave.
// The int32 accumulators go to S (FP64) every kFlush k tiles; a wave owns
// its output elements, so the first flush stores and later ones add, or, with
// the k range in shares (grid y), all add to the cleared S.
//
// Measured on the 768-histogram workload (768 x 16,384 bins x 8,192 q):
// operands loaded straight into registers kept the MFMA pipe busy 35% of
// the time, waiting on load latency (two waves per SIMD at 250 VGPRs, no
// registers for a prefetch); per-wave LDS stages one k tile ahead, with
// every wave fetching its own copy of the B tiles (9 KiB per wave per k
// tile), 50%.  Two waves side by side (WN = 2) load 14 KiB instead of 24 for the
// products of four waves: whole call with counts of one, two and three slices
// 916, 1,272 and 1,607 us (1,033, 1,397, 1,743 with WN = 1).
//
// BATCH: the column tiles come in groups of NT with their own k range and
// slices (tiles[tile0 + group]: the count slices at b_off, laid out
// [NB][NT][kt][64]), A is laid out with KT = the largest k range, and the
// columns go to the rows of S that cols[] names.  Otherwise all columns
// share KT and B is laid out [NB][NTn][KT][64].
template <int NA, int NB, int NT, int WN, bool BATCH>
__global__ __launch_bounds__(256 * WN, 2) void pairsum_mfma_lds_kernel(const v4i *__restrict__ As,
                                                                const v4i *__restrict__ Bs,
                                                                unsigned MT, unsigned NTn, unsigned KT,
                                                                unsigned nq, unsigned ncols,
                                                                double *__restrict__ S,
                                                                const MfmaTile *__restrict__ tiles,
                                                                const MfmaCol *__restrict__ cols,
                                                                unsigned tile0) {
  constexpr int DMIN = -(NA - 1);
  constexpr int DMAX = NB - 1;
  constexpr int NG = DMAX - DMIN + 1;
  constexpr int NBT = NB * NT * WN;    // B tiles per k tile
  constexpr int TPS = 4 * NA + NBT;    // tiles per stage
  constexpr int NW = 4 * WN;           // waves
  constexpr int NL = (TPS + NW - 1) / NW;  // of which a wave fetches at most NL
  constexpr int NS = 3;                // stages
  // loads per stage that every wave issues at least (the first waves issue one
  // more; waiting for this count still covers their older stage)
  constexpr int VM = TPS / NW;
  static_assert(VM <= 15, "vmcnt field");
  __shared__ v4i stage[NS][TPS][64];
  const unsigned lane = threadIdx.x & 63;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned wm = wave % 4, wn = wave / 4;
  const unsigned ngrp = NTn / (NT * WN);
  unsigned tile = blockIdx.x;
  if ((gridDim.x & 7u) == 0) tile = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const unsigned mg = tile / ngrp, ng = tile % ngrp;
  const unsigned mt = mg * 4 + wm;
  // this group's k tiles, B slice stride, B column-tile stride, B base
  unsigned KTg = KT;
  size_t sB = (size_t)NTn * KT * 64, tB = (size_t)KT * 64;
  const v4i *bp = Bs + (size_t)ng * NT * WN * KT * 64;
  unsigned col0 = (ng * WN + wn) * NT * 32, colend = ncols;
  if constexpr (BATCH) {
    static_assert(!BATCH || WN == 1, "a batch's groups are NT column tiles");
    const MfmaTile d = tiles[tile0 + ng];
    KTg = d.kt;
    sB = (size_t)NT * d.kt * 64;
    tB = (size_t)d.kt * 64;
    bp = Bs + d.b_off;
    col0 = d.col0;
    colend = min(ncols, d.col0 + d.ncol);
  }
  typedef __attribute__((address_space(3))) void lds_t;

  // the tiles of a stage go round the waves: the A tiles (q tile m, slice i) as
  // m NA + i, then the B tiles (slice j, column tile t) as 4 NA + j NT WN + t
  const v4i *src[NL];
#pragma unroll
  for (int l = 0; l < NL; ++l) {
    const int b = l * NW + (int)wave, c = b - 4 * NA;
    src[l] = c < 0 ? As + ((size_t)(b % NA) * MT + mg * 4 + b / NA) * KT * 64
                   : bp + (size_t)(c / (NT * WN)) * sB + (size_t)(c % (NT * WN)) * tB;
  }
  auto fetch = [&](unsigned kt, int st) {
#pragma unroll
    for (int l = 0; l < NL; ++l)
      if (l < TPS / NW || l * NW + (int)wave < TPS)
        __builtin_amdgcn_global_load_lds((const void *)(src[l] + (size_t)kt * 64 + lane),
                                         (lds_t *)&stage[st][l * NW + wave][0], 16, 0, 0);
  };
  // all waves: own LDS reads done, then the barrier; the empty asm keeps the
  // compiler from moving LDS accesses across it
  auto sync_lds = [&]() {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
  };

  // this share's k tiles
  const unsigned kfirst = (unsigned)((unsigned long long)KTg * blockIdx.y / gridDim.y);
  const unsigned klast = (unsigned)((unsigned long long)KTg * (blockIdx.y + 1) / gridDim.y);
  for (unsigned kb = kfirst; kb < klast; kb += kFlush) {
    const unsigned ke = min(klast, kb + kFlush);
    v16i acc[NG][NT];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[g][t] = v16i{0};
    // no wave still reads a stage of the previous block
    sync_lds();
    fetch(kb, 0);
    if (kb + 1 < ke) fetch(kb + 1, 1);
    int st = 0;
    for (unsigned kt = kb; kt < ke; ++kt) {
      if (kt + 1 < ke)
        __builtin_amdgcn_s_waitcnt(0x0f70 | VM);  // vmcnt(VM): own loads of stage kt landed
      else
        __builtin_amdgcn_s_waitcnt(0x0f70);       // vmcnt(0)
      sync_lds();
      if (kt + 2 < ke) fetch(kt + 2, st == 0 ? 2 : st - 1);
      v4i a[NA], b[NB][NT];
#pragma unroll
      for (int i = 0; i < NA; ++i) a[i] = stage[st][wm * NA + i][lane];
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) b[j][t] = stage[st][4 * NA + (j * WN + wn) * NT + t][lane];
#pragma unroll
      for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int t = 0; t < NT; ++t)
            acc[j - i - DMIN][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                BATCH ? a[i] : b[j][t], BATCH ? b[j][t] : a[i], acc[j - i - DMIN][t], 0, 0, 0);
      st = st == 2 ? 0 : st + 1;
    }
    auto value = [&](int t, int e) {
      double v = 0.0;
#pragma unroll
      for (int g = 0; g < NG; ++g) v = fma((double)acc[g][t][e], ldexp(1.0, 7 * (g + DMIN) - 6), v);
      return v;
    };
    // opaque, or the addresses would be formed before the loop over kb and kept
    unsigned stride = nq;
    __asm__ volatile("" : "+s"(stride));
    if constexpr (BATCH) {
      // lane % 32 is a column (one look at its row of S)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const unsigned col = col0 + t * 32 + (lane & 31);
        if (col >= colend) continue;
        const unsigned row0 = mt * 32 + 4 * (lane >> 5);
        double *const o0 = S + (size_t)cols[col].type * stride + row0;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const unsigned r = 8 * (e >> 2) + (e & 3);
          if (row0 + r < nq) {
            const double v = value(t, e);
            o0[r] = kb == 0 ? v : o0[r] + v;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else {
      // lane % 32 is a q, so that 32 lanes write 32 consecutive ones
      const unsigned row = mt * 32 + (lane & 31), cl = col0 + 4 * (lane >> 5);
      if (row >= nq) continue;
      double *const o0 = S + (size_t)cl * stride + row;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const unsigned c = t * 32 + 8 * (e >> 2) + (e & 3);
          if (cl + c < colend) {
            const double v = value(t, e);
            double *o = o0 + (size_t)c * stride;
            if (gridDim.y > 1)
              atomicAdd(o, v);
            else
              *o = kb == 0 ? v : *o + v;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
    }
  }
}

template <int NT, int WN, bool BATCH>
static void launch_gemm(int nb, dim3 grid, hipStream_t st, const v4i *As, const v4i *Bs, unsigned MT,
                        unsigned NTn, unsigned KT, unsigned nq, unsigned ncols, double *S,
                        const MfmaTile *tiles = nullptr, const MfmaCol *cols = nullptr,
                        unsigned tile0 = 0) {
#define XS_MM_LAUNCH(NBV, NTV)                                                                       \
  hipLaunchKernelGGL((pairsum_mfma_lds_kernel<kNA, NBV, NTV, WN, BATCH>), grid, dim3(256 * WN), 0, st, \
                     As, Bs, MT, NTn, KT, nq, ncols, S, tiles, cols, tile0)
  switch (nb) {
    case 1:
      XS_MM_LAUNCH(1, NT);
      break;
    case 2:
      XS_MM_LAUNCH(2, NT);
      break;
    case 3:
      if constexpr (NT == 1) XS_MM_LAUNCH(3, 1);  // three count slices with two column tiles would spill
      break;
    default:
      if constexpr (NT == 1) {
        if (nb == 4)
          XS_MM_LAUNCH(4, 1);
        else
          XS_MM_LAUNCH(5, 1);
      }
      break;
  }
#undef XS_MM_LAUNCH
}

}  // namespace mm

// Shares of the k range for `groups` work groups, `slots` of which run at a time: the
// rounds of work groups that a share takes, and the sums that every share adds to S
// (3% of the products of 512 k tiles).  Counts of two slices, 16,384 bins x 8,192 q,
// whole call: 768 histograms, a round and a half, 1,272 us in one share, 1,204 in two,
// 1,247 in three; 400, one round, 863 in one and 857 in two; 94, a quarter of one, 405
// in four and 462 in two.
static unsigned k_shares(unsigned groups, unsigned KT, unsigned slots) {
  unsigned best = 1;
  double cost = std::ceil((double)groups / slots);
  for (unsigned z = 2; z <= 16 && KT / z >= 32; ++z) {
    const double c = std::ceil((double)groups * z / slots) / z + 15.0 * z * groups / ((double)slots * KT);
    if (c < cost) {
      cost = c;
      best = z;
    }
  }
  return best;
}

int pairsum_mfma(xs_ctx *ctx, const unsigned long long *hist, unsigned ncols, unsigned nhist,
                 double bin, const double *q, unsigned nq, double *S) {
  using namespace mm;
  const unsigned MT = (nq + 127) / 128 * 4;
  const unsigned KT = (nhist + 31) / 32;
  const unsigned NTmax = (ncols + 127) / 128 * 4;  // column tiles for any form
  const size_t aBytes = (size_t)kNA * MT * KT * 1024, bBytes = (size_t)kMaxNB * NTmax * KT * 1024;
  XS_TRY(ensure_matrix(ctx, Carver::need({aBytes, bBytes, 8})));
  XS_TRY(ensure_pinned(ctx, 64));
  Carver cv(ctx->mat);
  v4i *As = cv.take<v4i>(aBytes / 16);
  v4i *Bs = cv.take<v4i>(bBytes / 16);
  unsigned long long *mx = cv.take<unsigned long long>(1);
  // bits of the largest count -> number of count slices (one read back, while the
  // sine's slices are made)
  const size_t hn = (size_t)ncols * nhist;
  hipLaunchKernelGGL(zero_u64, dim3(1), dim3(1), 0, ctx->stream, mx);
  hipLaunchKernelGGL(or_u64, dim3((unsigned)std::min<size_t>((hn + 1023) / 1024, 1024)), dim3(256), 0,
                     ctx->stream, hist, hn, mx);
  XS_HIP_CHECK(hipGetLastError());
  XS_HIP_CHECK(hipMemcpyAsync(ctx->pin, mx, 8, hipMemcpyDeviceToHost, ctx->stream));
  if (!ctx->read_back) XS_HIP_CHECK(hipEventCreateWithFlags(&ctx->read_back, hipEventDisableTiming));
  XS_HIP_CHECK(hipEventRecord(ctx->read_back, ctx->stream));
  hipEvent_t ev;
  XS_TRY(prof_begin(ctx, "pairsum_slices", &ev));
  launch_slice_sinc(ctx, q, nq, nhist, bin, MT, KT, As);
  XS_HIP_CHECK(hipGetLastError());
  XS_HIP_CHECK(hipEventSynchronize(ctx->read_back));
  const unsigned long long cmax = *static_cast<unsigned long long *>(ctx->pin);
  int nb = 1;
  while (nb < kMaxNB && (cmax >> (7 * nb)) != 0ull) ++nb;
  if ((cmax >> (7 * nb)) != 0ull) {
    XS_TRY(prof_end(ctx, "pairsum_slices", ev));
    return fail(XS_ERR_RANGE, "xs_hist_pairsum: a bin count exceeds 2^35 (matrix-core path)");
  }
  // two column tiles per wave unless the accumulators would not fit
  const int NT = (ncols > 32 && nb <= 2) ? 2 : 1;  // nb = 3 with NT = 2 would spill
  // two waves side by side where there are columns for both
  const int WN = ncols > 32u * NT ? 2 : 1;
  const unsigned NTn = (ncols + 32 * NT * WN - 1) / (32 * NT * WN) * (NT * WN);

  const size_t tb = (size_t)NTn * KT * 64;
  const unsigned groups = (MT / 4) * (NTn / (NT * WN));
  const unsigned shares = k_shares(groups, KT, 2 / WN * (unsigned)ctx->cu_count);
  hipLaunchKernelGGL(slice_counts, dim3((unsigned)((tb + 255) / 256)), dim3(256), 0, ctx->stream, hist,
                     ncols, nhist, NTn, KT, nb, Bs, shares > 1 ? S : nullptr, (size_t)ncols * nq);
  XS_HIP_CHECK(hipGetLastError());
  XS_TRY(prof_end(ctx, "pairsum_slices", ev));
  XS_TRY(prof_begin(ctx, "pairsum_mfma", &ev));
  const dim3 grid(groups, shares);
  auto gemm = [&](auto launch) {
    launch(nb, grid, ctx->stream, As, Bs, MT, NTn, KT, nq, ncols, S, nullptr, nullptr, 0u);
  };
  if (WN == 2 && NT == 2)
    gemm(launch_gemm<2, 2, false>);
  else if (WN == 2)
    gemm(launch_gemm<1, 2, false>);
  else if (NT == 2)
    gemm(launch_gemm<2, 1, false>);
  else
    gemm(launch_gemm<1, 1, false>);
  XS_HIP_CHECK(hipGetLastError());
  XS_TRY(prof_end(ctx, "pairsum_mfma", ev));
  return XS_OK;
}

int pairsum_mfma_batch(xs_ctx *ctx, const MfmaBatchPlan &plan, const unsigned long long *hist,
                       const MfmaCol *cols_d, const MfmaTile *tiles_d, void *a_buf, void *b_buf,
                       double bin, const double *q, unsigned nq, double *S, bool prof) {
  using namespace mm;
  if (nq != plan.nq) return fail(XS_ERR_ARG, "pairsum_mfma_batch: plan made for another nq");
  const unsigned MT = (nq + 127) / 128 * 4;
  const unsigned KT = plan.kt_max;
  const unsigned ncols = (unsigned)plan.cols.size();
  v4i *As = static_cast<v4i *>(a_buf), *Bs = static_cast<v4i *>(b_buf);
  hipEvent_t ev{};
  if (prof) XS_TRY(prof_begin(ctx, "batch_pairsum", &ev));
  launch_slice_sinc(ctx, q, nq, KT * 32, bin, MT, KT, As);
  for (const MfmaLaunch &L : plan.launches) {
    const size_t tb = (size_t)L.ntiles * L.nt * KT * 64;
    hipLaunchKernelGGL(slice_counts_batch, dim3((unsigned)((tb + 255) / 256)), dim3(256), 0,
                       ctx->stream, hist, cols_d, ncols, tiles_d, L.tile0, L.ntiles, KT, (int)L.nb,
                       (int)L.nt, Bs);
    const dim3 grid((MT / 4) * L.ntiles);
    if (L.nt == 2)
      launch_gemm<2, 1, true>((int)L.nb, grid, ctx->stream, As, Bs, MT, L.ntiles * 2, KT, nq, ncols, S,
                           tiles_d, cols_d, L.tile0);
    else
      launch_gemm<1, 1, true>((int)L.nb, grid, ctx->stream, As, Bs, MT, L.ntiles, KT, nq, ncols, S,
                           tiles_d, cols_d, L.tile0);
  }
  XS_HIP_CHECK(hipGetLastError());
  if (prof) XS_TRY(prof_end(ctx, "batch_pairsum", ev));
  return XS_OK;
}

}  // namespace xs
