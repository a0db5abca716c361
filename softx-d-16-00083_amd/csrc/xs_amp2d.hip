// H7: orientation-summed 2D intensity for an explicit q-vector list on gfx950.
//
// I[k] = sum_r | sum_el f_el(k) sum_{j in el} exp(i (R_r^T q_k) . x_j) |^2
// (CalcFunctions.cpp:1026-1062: the q vector is rotated by R^T instead of the
// atoms, 1020-1022 and 1033).
//
// One thread per (q point, rotation); the atoms stream through LDS in chunks
// of 256 (FP64 SoA), read by every lane at the same address (broadcast).
// The phase q'.x is formed in FP64 (in turns) and reduced to [0, 1), so the
// FP32 hardware sine and cosine (v_sin_f32 / v_cos_f32 take turns) see an
// argument accurate to 2^-24 turn even where q'.x reaches 10^2 turns; the
// element amplitudes are accumulated in FP64 and |A|^2 is added into the
// FP64 result with atomics (one per rotation and q point), or, where the atoms
// are given out in shares, the amplitudes are.  Bound by the issue of one term:
// three FMAs, v_fract_f64 (a floor and a subtraction took 5 cycles more), a
// conversion to FP32, two hardware sines, two conversions back and two adds,
// 53 cycles of a SIMD for 64 points, all of them issue; 20,000 atoms x 92,160
// points x 4 rotations 2.87 ms (3.11 with floor and one share).
#include <algorithm>
#include <cmath>

#include "xs_internal.h"
#include "xs_sincos.h"

namespace xs {
namespace amp2d {

constexpr int kBlock = 256;
constexpr int kChunk = 256;
constexpr double kInvTwoPi = 0.15915494309189533576888376337251;

struct Args {
  const double *x, *y, *z;
  const double *qvec;  // nqp x 3
  const double *rot;   // nrot x 9, row-major R
  const double *ff;    // n_el x nqp
  double *I;
  double *amp;  // nrot x nqp, complex
  unsigned nqp, n_el;
  unsigned el_off[17];
};

__global__ __launch_bounds__(kBlock) void amp2d_kernel(Args A) {
  __shared__ double sx[kChunk], sy[kChunk], sz[kChunk];
  const unsigned k = blockIdx.x * kBlock + threadIdx.x;
  const bool valid = k < A.nqp;
  const double *R = A.rot + 9 * (size_t)blockIdx.y;
  double qx = 0, qy = 0, qz = 0;
  if (valid) {
    const double a = A.qvec[3 * (size_t)k], b = A.qvec[3 * (size_t)k + 1],
                 c = A.qvec[3 * (size_t)k + 2];
    qx = (a * R[0] + b * R[3] + c * R[6]) * kInvTwoPi;
    qy = (a * R[1] + b * R[4] + c * R[7]) * kInvTwoPi;
    qz = (a * R[2] + b * R[5] + c * R[8]) * kInvTwoPi;
  }
  double Ar = 0.0, Ai = 0.0;
  unsigned chunk = 0;
  for (unsigned e = 0; e < A.n_el; ++e) {
    double ar = 0.0, ai = 0.0;
    const unsigned e0 = A.el_off[e], e1 = A.el_off[e + 1];
    for (unsigned c0 = e0; c0 < e1; c0 += kChunk) {
      if (chunk++ % gridDim.z != blockIdx.z) continue;
      const unsigned cn = min((unsigned)kChunk, e1 - c0);
      __syncthreads();
      for (unsigned j = threadIdx.x; j < cn; j += kBlock) {
        sx[j] = A.x[c0 + j];
        sy[j] = A.y[c0 + j];
        sz[j] = A.z[c0 + j];
      }
      __syncthreads();
#pragma unroll 4
      for (unsigned j = 0; j < cn; ++j) {
        const double ph = fma(qx, sx[j], fma(qy, sy[j], qz * sz[j]));
        const float f = (float)__builtin_amdgcn_fract(ph);
        ar += (double)__builtin_amdgcn_cosf(f);
        ai += (double)__builtin_amdgcn_sinf(f);
      }
    }
    if (valid) {
      const double w = A.ff[(size_t)e * A.nqp + k];
      Ar = fma(w, ar, Ar);
      Ai = fma(w, ai, Ai);
    }
  }
  if (!valid) return;
  if (gridDim.z > 1) {
    double *o = A.amp + 2 * ((size_t)blockIdx.y * A.nqp + k);
    atomicAdd(o, Ar);
    atomicAdd(o + 1, Ai);
  } else {
    atomicAdd(&A.I[k], Ar * Ar + Ai * Ai);
  }
}

// Regular q grid: q(iu, iv) = q0 + iu du + iv dv, point k = iv nu + iu, in runs
// of 16 consecutive points of a row.  For an atom x the phase advances by
// delta = (R^T du).x per point.  The run's first phase gives one FP32 hardware
// sine and cosine (FP64-reduced, as the list kernel), turned by 7.5 delta to the
// middle of the run in FP64; from there the points lie at +-b delta, b = 1/2 ...
// 15/2, so with z = C + i S of the middle
//   sum z e^{+-i b delta} = (sum C cos -+ sum S sin) + i (sum S cos +- sum C sin),
// two matrix products over the atoms, of 16 runs x (8 cosines, 8 sines) each, and
// every term serves both signs: 4 atoms x 16 runs x 16 points are two
// v_mfma_f64_16x16x4.  The cosines and sines of an atom are made once per work
// group and chunk (FP64, in LDS); a lane forms the seed of one run and atom, the
// layout that the instruction reads.
// Bound by the FP64 units: the matrix instructions (128 cycles of a SIMD for 64 runs
// and atoms) and the seeds (~65), which do not overlap.  50,000 atoms, 512 x 512
// points, 8 rotations: 9.3 ms; 16 points advanced one from another by a three-term
// recurrence (four FP64 operations a point, 330 cycles) took 16.1, and 10 times as
// long on planes of a few thousand runs, which left most of the chip idle.
constexpr int kRun = 16;
constexpr int kGridChunk = 128;

struct GridArgs {
  const double *x, *y, *z;
  const double *rot;  // nrot x 9
  const double *ff;   // n_el x nqp
  double *I;
  double *amp;  // nrot x nqp, complex
  double q0[3], du[3], dv[3];
  unsigned nu, nv, runs_per_row, n_el;
  unsigned el_off[17];
};

typedef double double4v __attribute__((ext_vector_type(4)));

// A wave has T tiles of 16 runs.  Grid (tiles, rotations, shares of the atoms'
// chunks): with more than one share the amplitudes are added up in A.amp.
template <int T>
__global__ __launch_bounds__(kBlock, T == 1 ? 4 : 3) void amp2d_grid_kernel(GridArgs A) {
  constexpr unsigned kStride = 17;  // of an atom's 16 columns: banks
  __shared__ double sx[kGridChunk], sy[kGridChunk], sz[kGridChunk], sb[kGridChunk * kStride];
  const unsigned lane = threadIdx.x & 63, col = lane & 15, kc = lane >> 4;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned run0 = (blockIdx.x * (kBlock / 64) + wave) * 16 * T;
  const double *R = A.rot + 9 * (size_t)blockIdx.y;
  // R^T applied to a vector, in turns
  auto turn = [&](double a, double b, double c, double *o) {
    o[0] = (a * R[0] + b * R[3] + c * R[6]) * kInvTwoPi;
    o[1] = (a * R[1] + b * R[4] + c * R[7]) * kInvTwoPi;
    o[2] = (a * R[2] + b * R[5] + c * R[8]) * kInvTwoPi;
  };
  double q[T][3], d[3];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const unsigned run = run0 + 16 * t + col;
    const unsigned iv = min(run / A.runs_per_row, A.nv - 1);
    const double u = (double)(run % A.runs_per_row * kRun), v = (double)iv;
    turn(A.q0[0] + u * A.du[0] + v * A.dv[0], A.q0[1] + u * A.du[1] + v * A.dv[1],
         A.q0[2] + u * A.du[2] + v * A.dv[2], q[t]);
  }
  turn(A.du[0], A.du[1], A.du[2], d);
  // the lane's points: run run0 + 16 t + kc + 4 i, place 8 + col or, from column 8
  // on, 15 - col
  const bool low = col < 8;
  const unsigned place = low ? 8 + col : 15 - col;
  double Ar[T][4], Ai[T][4];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) Ar[t][i] = Ai[t][i] = 0.0;
  auto point = [&](int t, int i, size_t *k) {
    const unsigned run = run0 + 16 * t + kc + 4 * i, iv = run / A.runs_per_row;
    const unsigned iu = run % A.runs_per_row * kRun + place;
    *k = (size_t)iv * A.nu + iu;
    return iv < A.nv && iu < A.nu;
  };
  unsigned chunk = 0;
  for (unsigned e = 0; e < A.n_el; ++e) {
    double4v ac[T], as[T];
#pragma unroll
    for (int t = 0; t < T; ++t) ac[t] = as[t] = (double4v){0.0, 0.0, 0.0, 0.0};
    const unsigned e0 = A.el_off[e], e1 = A.el_off[e + 1];
    for (unsigned c0 = e0; c0 < e1; c0 += kGridChunk) {
      if (chunk++ % gridDim.z != blockIdx.z) continue;
      const unsigned cn = min((unsigned)kGridChunk, e1 - c0);
      __syncthreads();
      {  // two threads an atom, four of b each; atoms beyond the last are zeros
        const unsigned j = threadIdx.x % kGridChunk, half = threadIdx.x / kGridChunk;
        const bool in = j < cn;
        const double xj = in ? A.x[c0 + j] : 0.0, yj = in ? A.y[c0 + j] : 0.0,
                     zj = in ? A.z[c0 + j] : 0.0;
        if (half == 0) {
          sx[j] = xj;
          sy[j] = yj;
          sz[j] = zj;
        }
        const double st = fma(d[0], xj, fma(d[1], yj, d[2] * zj));
        double sn, cs, s1, c1;
        sincos_2pi(st, &s1, &c1);
        sincos_2pi((half ? 4.5 : 0.5) * (st - rint(0.5 * st) * 2.0), &sn, &cs);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          sb[j * kStride + 4 * half + b] = in ? cs : 0.0;
          sb[j * kStride + 8 + 4 * half + b] = in ? sn : 0.0;
          const double c = fma(cs, c1, -(sn * s1));
          sn = fma(cs, s1, sn * c1);
          cs = c;
        }
      }
      __syncthreads();
      for (unsigned j0 = 0; j0 < cn; j0 += 4) {
        const unsigned j = j0 + kc;
        const double xj = sx[j], yj = sy[j], zj = sz[j];
        const double b = sb[j * kStride + col], rc = sb[j * kStride + 7], rs = sb[j * kStride + 15];
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const double ph = fma(q[t][0], xj, fma(q[t][1], yj, q[t][2] * zj));
          const float f = (float)__builtin_amdgcn_fract(ph);
          const double c = (double)__builtin_amdgcn_cosf(f), s = (double)__builtin_amdgcn_sinf(f);
          ac[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(fma(c, rc, -(s * rs)), b, ac[t], 0, 0, 0);
          as[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(fma(s, rc, c * rs), b, as[t], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // columns 0-7: sum C cos, sum S cos; 8-15: sum C sin, sum S sin
        const double pc = __shfl_xor(ac[t][i], 8, 64), ps = __shfl_xor(as[t][i], 8, 64);
        const double re = low ? ac[t][i] - ps : pc + as[t][i];
        const double im = low ? as[t][i] + pc : ps - ac[t][i];
        size_t k;
        if (point(t, i, &k)) {
          const double w = A.ff[(size_t)e * A.nu * A.nv + k];
          Ar[t][i] = fma(w, re, Ar[t][i]);
          Ai[t][i] = fma(w, im, Ai[t][i]);
        }
      }
  }
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      size_t k;
      if (!point(t, i, &k)) continue;
      if (gridDim.z > 1) {
        double *o = A.amp + 2 * ((size_t)blockIdx.y * A.nu * A.nv + k);
        atomicAdd(o, Ar[t][i]);
        atomicAdd(o + 1, Ai[t][i]);
      } else {
        atomicAdd(&A.I[k], Ar[t][i] * Ar[t][i] + Ai[t][i] * Ai[t][i]);
      }
    }
}

__global__ void sum_squares(const double *__restrict__ amp, size_t nqp, unsigned nrot,
                            double *__restrict__ I) {
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < nqp;
       k += (size_t)gridDim.x * blockDim.x) {
    double v = 0.0;
    for (unsigned r = 0; r < nrot; ++r) {
      const double *a = amp + 2 * (r * nqp + k);
      v += a[0] * a[0] + a[1] * a[1];
    }
    I[k] = v;
  }
}

__global__ void zero_f64(double *__restrict__ p, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0.0;
}

// How many shares the atoms are given out in.  Few work groups leave CUs idle or a
// last round of them nearly empty: below 8 a CU the atoms are shared out until there
// are 12, two chunks a share at least.  Not under stream capture, where a graph would
// keep the scratch's address, nor without memory for the amplitudes.
// Grid, 31,170 atoms, 304 x 240 points, 8 rotations: 2.0 ms (one share 2.5); 32,397
// atoms, 363 x 375, 8 rotations: 3.7 ms (one share, tiles in pairs: 4.6).  List, 20,000
// atoms, 92,160 points, 4 rotations: 2.87 ms; 10,106 atoms, 6,319 points, 2 rotations:
// 65 us (one share 387).
static int atom_shares(xs_ctx *ctx, size_t groups, size_t n_atoms, unsigned chunk, size_t amplitudes,
                       unsigned *shares) {
  *shares = 1;
  const size_t most = (n_atoms + chunk - 1) / chunk / 2, cus = (size_t)ctx->cu_count;
  if (groups >= 8 * cus || most < 2) return XS_OK;
  hipStreamCaptureStatus capture;
  XS_HIP_CHECK(hipStreamIsCapturing(ctx->stream, &capture));
  if (capture != hipStreamCaptureStatusNone) return XS_OK;
  const size_t want = std::min<size_t>(std::min(12 * cus / groups, most), 65535);
  if (want < 2) return XS_OK;
  const int e = ensure_matrix(ctx, amplitudes * 16);
  if (e == XS_OK) *shares = (unsigned)want;
  return e == XS_ERR_NOMEM ? XS_OK : e;
}

}  // namespace amp2d
}  // namespace xs

using namespace xs;

extern "C" int xs_amp2d(xs_ctx *ctx, const double *xyz, size_t n_atoms, const unsigned *el_count,
                        unsigned n_el, const double *qvec, size_t nqp, const double *rot,
                        unsigned nrot, const double *ff, double *I, unsigned flags) {
  XS_TRY(activate(ctx));
  if (!el_count || !qvec || !rot || !ff || !I || (!xyz && n_atoms))
    return fail(XS_ERR_ARG, "xs_amp2d: null pointer");
  if (n_el == 0 || n_el > 16) return fail(XS_ERR_RANGE, "xs_amp2d: n_el must be in [1, 16]");
  size_t tot = 0;
  for (unsigned e = 0; e < n_el; ++e) tot += el_count[e];
  if (tot != n_atoms) return fail(XS_ERR_ARG, "xs_amp2d: sum(el_count) != n_atoms");
  if (n_atoms >= (size_t(1) << 32) || nqp >= (size_t(1) << 31))
    return fail(XS_ERR_RANGE, "xs_amp2d: size too large");
  if (nqp == 0) return XS_OK;
  if (nrot == 0 || nrot > 65535) return fail(XS_ERR_RANGE, "xs_amp2d: nrot must be in [1, 65535]");
  const bool device = flags & XS_DEVICE_PTRS;
  amp2d::Args A{};
  A.nqp = (unsigned)nqp;
  A.n_el = n_el;
  A.el_off[0] = 0;
  for (unsigned e = 0; e < n_el; ++e) A.el_off[e + 1] = A.el_off[e] + el_count[e];
  const double *xyzd = xyz, *qd = qvec, *rd = rot, *fd = ff;
  double *Id = I;
  if (!device) {
    XS_TRY(ensure_workspace(ctx, Carver::need({3 * n_atoms * 8, 3 * nqp * 8, (size_t)nrot * 72,
                                               (size_t)n_el * nqp * 8, nqp * 8})));
    Carver cv(ctx->ws);
    double *x2 = cv.take<double>(3 * n_atoms), *q2 = cv.take<double>(3 * nqp),
           *r2 = cv.take<double>((size_t)nrot * 9), *f2 = cv.take<double>((size_t)n_el * nqp);
    Id = cv.take<double>(nqp);
    XS_HIP_CHECK(hipMemcpyAsync(x2, xyz, 3 * n_atoms * 8, hipMemcpyHostToDevice, ctx->stream));
    XS_HIP_CHECK(hipMemcpyAsync(q2, qvec, 3 * nqp * 8, hipMemcpyHostToDevice, ctx->stream));
    XS_HIP_CHECK(hipMemcpyAsync(r2, rot, (size_t)nrot * 72, hipMemcpyHostToDevice, ctx->stream));
    XS_HIP_CHECK(hipMemcpyAsync(f2, ff, (size_t)n_el * nqp * 8, hipMemcpyHostToDevice, ctx->stream));
    xyzd = x2;
    qd = q2;
    rd = r2;
    fd = f2;
  }
  A.x = xyzd;
  A.y = xyzd + n_atoms;
  A.z = xyzd + 2 * n_atoms;
  A.qvec = qd;
  A.rot = rd;
  A.ff = fd;
  A.I = Id;
  const size_t groups = (nqp + amp2d::kBlock - 1) / amp2d::kBlock;
  unsigned shares = 1;
  XS_TRY(amp2d::atom_shares(ctx, groups * nrot, n_atoms, amp2d::kChunk, (size_t)nrot * nqp, &shares));
  A.amp = static_cast<double *>(ctx->mat);
  double *const sum = shares > 1 ? A.amp : Id;
  const size_t nsum = shares > 1 ? 2 * (size_t)nrot * nqp : nqp;
  hipLaunchKernelGGL(amp2d::zero_f64, dim3((unsigned)std::min<size_t>((nsum + 255) / 256, 4096)),
                     dim3(256), 0, ctx->stream, sum, nsum);
  hipEvent_t ev;
  XS_TRY(prof_begin(ctx, "amp2d", &ev));
  hipLaunchKernelGGL(amp2d::amp2d_kernel, dim3((unsigned)groups, nrot, shares), dim3(amp2d::kBlock), 0,
                     ctx->stream, A);
  if (shares > 1)
    hipLaunchKernelGGL(amp2d::sum_squares, dim3((unsigned)std::min<size_t>((nqp + 255) / 256, 4096)),
                       dim3(256), 0, ctx->stream, A.amp, nqp, nrot, Id);
  XS_HIP_CHECK(hipGetLastError());
  XS_TRY(prof_end(ctx, "amp2d", ev));
  if (!device) {
    XS_HIP_CHECK(hipMemcpyAsync(I, Id, nqp * 8, hipMemcpyDeviceToHost, ctx->stream));
    XS_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  }
  return XS_OK;
}

extern "C" int xs_amp2d_grid(xs_ctx *ctx, const double *xyz, size_t n_atoms,
                             const unsigned *el_count, unsigned n_el, const double *q0,
                             const double *du, const double *dv, unsigned nu, unsigned nv,
                             const double *rot, unsigned nrot, const double *ff, double *I,
                             unsigned flags) {
  XS_TRY(activate(ctx));
  if (!el_count || !q0 || !du || !dv || !rot || !ff || !I || (!xyz && n_atoms))
    return fail(XS_ERR_ARG, "xs_amp2d_grid: null pointer");
  if (n_el == 0 || n_el > 16) return fail(XS_ERR_RANGE, "xs_amp2d_grid: n_el must be in [1, 16]");
  size_t tot = 0;
  for (unsigned e = 0; e < n_el; ++e) tot += el_count[e];
  if (tot != n_atoms) return fail(XS_ERR_ARG, "xs_amp2d_grid: sum(el_count) != n_atoms");
  const size_t nqp = (size_t)nu * nv;
  if (n_atoms >= (size_t(1) << 32) || nqp >= (size_t(1) << 31))
    return fail(XS_ERR_RANGE, "xs_amp2d_grid: size too large");
  if (nqp == 0) return XS_OK;
  if (nrot == 0 || nrot > 65535)
    return fail(XS_ERR_RANGE, "xs_amp2d_grid: nrot must be in [1, 65535]");
  const bool device = flags & XS_DEVICE_PTRS;
  amp2d::GridArgs A{};
  A.nu = nu;
  A.nv = nv;
  A.runs_per_row = (nu + amp2d::kRun - 1) / amp2d::kRun;
  A.n_el = n_el;
  for (int k = 0; k < 3; ++k) {
    A.q0[k] = q0[k];
    A.du[k] = du[k];
    A.dv[k] = dv[k];
  }
  A.el_off[0] = 0;
  for (unsigned e = 0; e < n_el; ++e) A.el_off[e + 1] = A.el_off[e] + el_count[e];
  const double *xyzd = xyz, *rd = rot, *fd = ff;
  double *Id = I;
  if (!device) {
    XS_TRY(ensure_workspace(ctx, Carver::need({3 * n_atoms * 8, (size_t)nrot * 72,
                                               (size_t)n_el * nqp * 8, nqp * 8})));
    Carver cv(ctx->ws);
    double *x2 = cv.take<double>(3 * n_atoms), *r2 = cv.take<double>((size_t)nrot * 9),
           *f2 = cv.take<double>((size_t)n_el * nqp);
    Id = cv.take<double>(nqp);
    XS_HIP_CHECK(hipMemcpyAsync(x2, xyz, 3 * n_atoms * 8, hipMemcpyHostToDevice, ctx->stream));
    XS_HIP_CHECK(hipMemcpyAsync(r2, rot, (size_t)nrot * 72, hipMemcpyHostToDevice, ctx->stream));
    XS_HIP_CHECK(hipMemcpyAsync(f2, ff, (size_t)n_el * nqp * 8, hipMemcpyHostToDevice, ctx->stream));
    xyzd = x2;
    rd = r2;
    fd = f2;
  }
  A.x = xyzd;
  A.y = xyzd + n_atoms;
  A.z = xyzd + 2 * n_atoms;
  A.rot = rd;
  A.ff = fd;
  A.I = Id;
  const size_t tiles = ((size_t)A.runs_per_row * nv + 15) / 16, groups = (tiles + 3) / 4 * nrot;
  // (two tiles a wave share the loads of an atom: 9.3 ms for 50,000 atoms, 512 x 512
  // points and 8 rotations, 9.8 with one; more than that loses to shares below it)
  unsigned shares = 1;
  XS_TRY(amp2d::atom_shares(ctx, groups, n_atoms, amp2d::kGridChunk, (size_t)nrot * nqp, &shares));
  A.amp = static_cast<double *>(ctx->mat);
  double *const sum = shares > 1 ? A.amp : Id;
  const size_t nsum = shares > 1 ? 2 * (size_t)nrot * nqp : nqp;
  hipLaunchKernelGGL(amp2d::zero_f64, dim3((unsigned)std::min<size_t>((nsum + 255) / 256, 4096)),
                     dim3(256), 0, ctx->stream, sum, nsum);
  hipEvent_t ev;
  XS_TRY(prof_begin(ctx, "amp2d", &ev));
  if (groups >= 8 * (size_t)ctx->cu_count)
    hipLaunchKernelGGL(amp2d::amp2d_grid_kernel<2>, dim3((unsigned)((tiles + 7) / 8), nrot),
                       dim3(amp2d::kBlock), 0, ctx->stream, A);
  else
    hipLaunchKernelGGL(amp2d::amp2d_grid_kernel<1>, dim3((unsigned)((tiles + 3) / 4), nrot, shares),
                       dim3(amp2d::kBlock), 0, ctx->stream, A);
  if (shares > 1)
    hipLaunchKernelGGL(amp2d::sum_squares, dim3((unsigned)std::min<size_t>((nqp + 255) / 256, 4096)),
                       dim3(256), 0, ctx->stream, A.amp, nqp, nrot, Id);
  XS_HIP_CHECK(hipGetLastError());
  XS_TRY(prof_end(ctx, "amp2d", ev));
  if (!device) {
    XS_HIP_CHECK(hipMemcpyAsync(I, Id, nqp * 8, hipMemcpyDeviceToHost, ctx->stream));
    XS_HIP_CHECK(hipStreamSynchronize(ctx->stream));
  }
  return XS_OK;
}
