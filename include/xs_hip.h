/*
 * xs_hip.h -- C ABI of the MI355X (gfx950) backend for the XaNSoNS
 * scattering calculators.
 *
 * The reference picks its calculator backend at link time: main.cpp declares
 * one set of prototypes (CPU main.cpp:65-68, CUDA main.cpp:46-52, OpenCL
 * main.cpp:54-63) and calls one of them per scenario (main.cpp:151-233).
 * This library is what a HIP build links instead.  The C++ drop-in
 * (softx-d-16-00083_amd/dropin/CalcFunctionsHIP.cpp) keeps the CPU
 * signatures of main.cpp:65-68 and calls the functions below; the Python
 * harness binds the same symbols with ctypes.
 *
 * Conventions
 *  - Every call returns XS_OK (0) or a negative XS_ERR_* code; the message
 *    of the last failure on the calling thread is xs_last_error().
 *  - Coordinates are structure-of-arrays: xyz[0..n) x, [n..2n) y, [2n..3n) z,
 *    atoms grouped element-major (el_count[0] atoms of element 0 first, ...).
 *  - el_count, and every scalar, is host memory.  The array arguments are
 *    host memory (the call copies, computes and returns synchronously) or,
 *    with XS_DEVICE_PTRS, device memory on the context's device (the call
 *    enqueues on the context stream and returns without waiting).
 *  - Pair types p = (a <= b) are ordered (0,0),(0,1),...,(0,n-1),(1,1),...
 *    (CalcFunctions.cpp:777-778); ntypes = n_el*(n_el+1)/2.
 *  - One context per host thread; calls on one context are serialised on
 *    its stream.
 */
#ifndef XS_HIP_H
#define XS_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define XS_OK 0
#define XS_ERR_ARG (-1)     /* invalid argument */
#define XS_ERR_HIP (-2)     /* a HIP runtime call failed */
#define XS_ERR_NOMEM (-3)   /* device or pinned allocation failed */
#define XS_ERR_DEVICE (-4)  /* no usable device / bad device id */
#define XS_ERR_RANGE (-5)   /* a size exceeds what the kernels support */

/* flags */
#define XS_DEVICE_PTRS 0x1u     /* array arguments are device pointers */
#define XS_F64_BINNING 0x2u     /* xs_hist: xyz is double, bin as the CPU path (double) */
#define XS_PDF_CPU_RADIUS 0x4u  /* xs_pdf: radius offset of the CPU path for p >= 1 */
#define XS_BATCH_GRAPH 0x8u     /* xs_batch_run: capture once, replay as a hipGraph */
#define XS_PAIRSUM_MFMA 0x10u   /* xs_hist_pairsum: int8 matrix-core product */
#define XS_F32_DOUBLE_QUOTIENT 0x20u /* xs_hist, xs_batch_plan, FP32 binning: skip the
                                        FP32 quotient form (see xs_hist) */
#define XS_PAIRSUM_F32 0x40u    /* xs_hist_pairsum: plain FP32 terms and sums (comparison) */

/* PDF types, typedefs.h:54-56 */
#define XS_PDF_RDF 0
#define XS_PDF_PDF 1
#define XS_PDF_RPDF 2

typedef struct xs_ctx xs_ctx;
typedef struct xs_batch xs_batch;
typedef struct xs_atoms xs_atoms;

/* Open a context on a device and create its stream.
 * Replaces SetDeviceCuda (CalcFunctionsCUDA.cu:1485-1519), which falls back
 * to the fastest device on a bad id; here a bad id is XS_ERR_DEVICE. */
int xs_init(int device, xs_ctx **ctx);

/* Release the context, its stream and workspace.
 * Replaces delDataFromDevice (CalcFunctionsCUDA.cu:1557-1566). */
int xs_free(xs_ctx *ctx);

/* Use an existing HIP stream (hipStream_t) for all later calls; NULL
 * restores the context's own stream.  No counterpart in the reference
 * (its calls are synchronous on the null stream). */
int xs_set_stream(xs_ctx *ctx, void *stream);

/* Wait for all work enqueued on the context stream. */
int xs_synchronize(xs_ctx *ctx);

/* Message of the last failure on this thread ("" if none). */
const char *xs_last_error(void);

/* Number of visible HIP devices. */
int xs_device_count(int *count);

/* Per-kernel timing with HIP events on the context stream.  enable=1 starts
 * (and resets) collection; xs_profile_read waits for the recorded events and
 * returns the summed duration and launch count of one kernel family:
 * "hist", "hist_prep", "hist_pairsum", "pdf", "debye", "amp2d".
 * Replaces the commented-out per-kernel cudaEvent timers
 * (CalcFunctionsCUDA.cu:716-731, 899-909, 1016-1032). */
int xs_profile(xs_ctx *ctx, int enable);
int xs_profile_read(xs_ctx *ctx, const char *kernel, double *total_ms,
                    unsigned long long *count);

/* H1: per-pair-type histogram of interatomic distances (uint64 counts).
 * Default: xyz is float and the bin index is (unsigned)(sqrtf((dx*dx+dy*dy)
 * +dz*dz)/bin) in IEEE single precision, the expression of calcHistKernel
 * (CalcFunctionsCUDA.cu:832-833) without fast-math.  With XS_F64_BINNING xyz
 * is double and the index is computed in double exactly as calcHist does
 * (CalcFunctions.cpp:784-788), so the counts equal the reference CPU path's.
 * Same-element pairs are j > i, cross-element pairs all (i, j)
 * (CalcFunctions.cpp:782).  hist (ntypes*nhist) is overwritten; pairs whose
 * index is >= nhist go to *overflow (may be NULL; with XS_DEVICE_PTRS a
 * device pointer).  FP32 binning evaluates the IEEE quotient by bin either as
 * a rounded double product or, for a bin width that a check over all 2^23
 * significands has passed (once per bin and context; it synchronises), with
 * FP32 operations only, which is faster; XS_F32_DOUBLE_QUOTIENT keeps the
 * double product.  Both give the IEEE quotient, so the counts are the same.
 * Host arrays pass through a device buffer that the context keeps until
 * xs_free (3 * n_atoms coordinates and ntypes * nhist counts); the work
 * between the copies is that of a device-pointer call.
 * Replaces calcHist (CalcFunctions.cpp:757-809) and calcHistCuda
 * (CalcFunctionsCUDA.cu:855-920). */
int xs_hist(xs_ctx *ctx, const void *xyz, size_t n_atoms,
            const unsigned *el_count, unsigned n_el, double bin, unsigned nhist,
            uint64_t *hist, uint64_t *overflow, unsigned flags);

/* H3: histogram pair sums S[p*nq+iq] = sum_k h_p[k] sin(q r_k)/(q r_k + 1e-8),
 * r_k = (k+1/2) bin, S = 0 where q = 0.  FP64: groups of bins act through 64
 * Chebyshev nodes each, to FP64 rounding (every bin by itself where they are
 * wider than ~0.6 / max |q|); the sums over the nodes are matrix products.
 * Up to 384 bins are summed bin by bin where that is faster.
 * Replaces the bin loop of calcInt1DHist (CalcFunctions.cpp:844-871) and
 * calcIntHistKernelXray/Neutron (CalcFunctionsCUDA.cu:923-985).
 * XS_PAIRSUM_MFMA evaluates the same sums as one product S = H A^T on the
 * int8 matrix cores: A (the sinc table) split into five int8 slices, the
 * counts into exact 7-bit slices, int32 accumulation; the result differs
 * from the FP64 sum by about 2^-35 sum_k h[k] (needs counts < 2^35 and a
 * workspace of ~5 nq nhist bytes, and reads the counts' extents back).  The
 * flag chooses the arithmetic, not the faster form: where 64 nodes stand for
 * more than ~300 bins the FP64 form is faster.
 * On device arrays and without XS_PAIRSUM_MFMA the call may be captured: it
 * then sums bin by bin, without scratch (as it does where the node tables'
 * memory, at most ~260 MiB + 16 bytes a bin, cannot be had).
 * XS_PAIRSUM_F32 evaluates the terms and the sums over 2048-bin chunks in
 * FP32 (IEEE sinf), the arithmetic of the reference GPU kernels; its error
 * against FP64 reaches ~1e-4 of I(q) at low q, where I(q) is a cancelling
 * difference, so it is there for comparison, not for results. */
int xs_hist_pairsum(xs_ctx *ctx, const uint64_t *hist, unsigned ntypes,
                    unsigned nhist, double bin, const double *q, unsigned nq,
                    double *S, unsigned flags);

/* H4: RDF / PDF / rPDF from the histogram in FP64, pdf = (1+ntypes)*nhist,
 * total first.  Replaces CalcFunctions.cpp:919-957 and
 * CalcFunctionsCUDA.cu:1092-1150.  XS_PDF_CPU_RADIUS reproduces the CPU
 * loop's radius r = (p*nhist + k + 1/2) bin for pair types p >= 1
 * (CalcFunctions.cpp:942, 950); without it r = (k + 1/2) bin as the CUDA
 * and OpenCL kernels compute (CalcFunctionsCUDA.cu:1057, 1066). */
int xs_pdf(xs_ctx *ctx, const uint64_t *hist, unsigned n_el,
           const unsigned *el_count, unsigned nhist, double bin, int pdf_type,
           double rho0, const double *sl, double *pdf, unsigned flags);

/* H5: direct Debye pair sums S[p*nq+iq] = sum_{pairs in p} sin(q r)/(q r + 1e-8)
 * with FP64 pair terms (xyz double).  Where that is cheaper the sums go
 * through Chebyshev moments of the pair distances, to the FP64 rounding of a
 * pair's term; else, on a uniform q mesh (the reference's,
 * ReadXML.cpp:220-222) sin(q r) advances from q to q by a recurrence, and
 * other meshes evaluate the series per q.
 * Replaces the pair loop of calcIntDebye (CalcFunctions.cpp:561-591) and
 * calcIntDebyeKernel (CalcFunctionsCUDA.cu:1163-1273). */
int xs_debye_pairsum(xs_ctx *ctx, const double *xyz, size_t n_atoms,
                     const unsigned *el_count, unsigned n_el, const double *q,
                     unsigned nq, double *S, unsigned flags);

/* Allocation-free variant of xs_debye_pairsum, for callers that cannot
 * allocate device memory (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc).  No counterpart in the reference.
 * xyz, q and S are device pointers (flags must hold XS_DEVICE_PTRS); the call
 * enqueues on the context stream and returns without waiting.  It calls no
 * hipMalloc/hipFree, no memset and no host copy: the kernels' tile and
 * work-item tables are built on the device in a 32 MiB scratch array that
 * the library holds on every device it runs on until the process ends.
 * Limit: the tables of the structure must fit the scratch -- 16 bytes per
 * tile of 32 atoms and per tile pair, about 65,000 atoms; larger inputs get
 * XS_ERR_RANGE (use xs_debye_pairsum).  Every call on a device shares its
 * scratch: calls that overlap on one device (several streams or threads)
 * race, so serialise them. */
int xs_debye_pairsum_noalloc(xs_ctx *ctx, const double *xyz, size_t n_atoms,
                             const unsigned *el_count, unsigned n_el, const double *q,
                             unsigned nq, double *S, unsigned flags);

/* H6: block-pair partial Debye sums.  blk_count[el*nblocks+b] atoms of
 * element el belong to block b (block-major inside each element).
 * S[(p*nparts + part)*nq + iq], part(iB<=jB) = nblocks*iB - iB*(iB+1)/2 + jB.
 * Replaces the pair loop of calcIntPartialDebye (CalcFunctions.cpp:662-703). */
int xs_partial_debye_pairsum(xs_ctx *ctx, const double *xyz, size_t n_atoms,
                             const unsigned *el_count, unsigned n_el,
                             const unsigned *blk_count, unsigned nblocks,
                             const double *q, unsigned nq, double *S,
                             unsigned flags);

/* H7: orientation-summed squared amplitude for an explicit q-vector list,
 * I[k] = sum_r | sum_el ff[el*nqp+k] sum_{j in el} exp(i (R_r^T q_k).x_j) |^2,
 * rot[r*9..] = R_r row-major (all double).  FP64 phase q'.x reduced to one
 * turn, FP32 hardware sin/cos of the reduced phase, FP64 amplitude sums.
 * Replaces calcInt2DKernelXray/Neutron + Sum2DKernel
 * (CalcFunctionsCUDA.cu:514-650) and the inner loops of calcInt2D
 * (CalcFunctions.cpp:1026-1062). */
int xs_amp2d(xs_ctx *ctx, const double *xyz, size_t n_atoms,
             const unsigned *el_count, unsigned n_el, const double *qvec,
             size_t nqp, const double *rot, unsigned nrot, const double *ff,
             double *I, unsigned flags);

/* H7 on a regular q grid: q(iu, iv) = q0 + iu du + iv dv (iu < nu, iv < nv),
 * point k = iv*nu + iu; otherwise as xs_amp2d (ff[el*nu*nv + k], I[k]).
 * Along a row the phase of an atom advances by (R^T du).x per point, so a
 * run of 16 points takes one FP32 hardware sine/cosine of the FP64-reduced
 * phase (the list kernel's accuracy), turned to the run's middle in FP64; the
 * sums over the atoms of its product with the sines and cosines of the
 * points' steps from there are FP64 matrix products.  q0, du, dv are host
 * arrays of 3; the rest as xs_amp2d.  The Cartesian q planes of 2D patterns
 * are such grids; the reference's polar (q, phi) mesh is not (use xs_amp2d). */
int xs_amp2d_grid(xs_ctx *ctx, const double *xyz, size_t n_atoms, const unsigned *el_count,
                  unsigned n_el, const double *q0, const double *du, const double *dv,
                  unsigned nu, unsigned nv, const double *rot, unsigned nrot, const double *ff,
                  double *I, unsigned flags);

/* Cut-off pair sums of RearrangementInt (CalcFunctions.cpp:485-499):
 * S[(el[i]*n_el + el[j])*nq + iq] = sum over ordered pairs (i, j) with
 * 1e-6 < r_ij^2 < rmax2[i] of sin(q r_ij)/(q r_ij + 1e-8), r_ij^2 =
 * (dx^2 + dy^2) + dz^2 in FP64 as the reference computes it (so the same
 * pairs are accepted); npairs[el[i]*n_el + el[j]] counts them.  xyz is SoA
 * (n_atoms), el[i] < n_el <= 64.  S (n_el^2 * nq) and npairs (n_el^2) are
 * overwritten.  Host arrays only (synchronous).  Replaces the pair loop of
 * RearrangementInt; its caller keeps the weighting and normalisation. */
int xs_cutoff_pairsum(xs_ctx *ctx, const double *xyz, size_t n_atoms, const unsigned *el,
                      unsigned n_el, const double *rmax2, const double *q, unsigned nq,
                      double *S, uint64_t *npairs, unsigned flags);

/* Sine sums over a list of distances: S[type[p]*nq + iq] = sum_p
 * sin(q r_p)/(q r_p + 1e-8), S (ntypes * nq) overwritten.  Host arrays only
 * (synchronous).  Replaces the neighbour loop of RearrangementInt
 * (CalcFunctions.cpp:506-529). */
int xs_pairlist_pairsum(xs_ctx *ctx, const double *r, const unsigned *type, size_t npairs,
                        unsigned ntypes, const double *q, unsigned nq, double *S,
                        unsigned flags);

/* Ensembles.  The reference computes one structure per run of main
 * (main.cpp:151-233: calcPDFandDebye per configuration); an ensemble of
 * particles is a sequence of such runs.  A batch plan holds every structure
 * on the device so that one xs_batch_run computes all of them.
 *
 * xs_batch_plan: structure s has n_el[s] elements; its el_count entries
 * follow those of structure s-1 in el_count; xyz[s] is its element-major
 * double SoA (3 * N_s values, host memory).  Coordinates are binned in double
 * with XS_F64_BINNING (calcHist, CalcFunctions.cpp:784-788), else rounded to
 * float and binned as calcHistKernel (CalcFunctionsCUDA.cu:832-833), with
 * the quotient form chosen as in xs_hist (XS_F32_DOUBLE_QUOTIENT applies).
 * nhist[s] = 0 (or nhist == NULL) takes GetHistSize's bin count
 * (CalcFunctions.cpp:224-243).  Each structure needs at least one atom.
 * With XS_DEVICE_PTRS the xyz[s] are device pointers (the array xyz itself
 * is host memory) and the structures are tiled on the GPU (all atoms at
 * once; fewer than 2^31 atoms in all); otherwise they are
 * tiled on the host's cores and uploaded.  Either way the call returns
 * when the plan is ready, and the coordinates are not needed afterwards.
 * The plan holds on the device the sorted coordinates (24 or 12 bytes per
 * atom), the tile tables and, for FP64 binning, 32 bytes of J records per
 * atom (each atom relative to its tile's centre). */
int xs_batch_plan(xs_ctx *ctx, unsigned nstruct, const unsigned *n_el,
                  const unsigned *el_count, const double *const *xyz,
                  double bin, const unsigned *nhist, unsigned flags,
                  xs_batch **plan);

/* Layout of a plan's outputs.  Structure s: histograms at hist_off[s]
 * (ntypes_s * nhist[s] bins), PDFs at pdf_off[s] ((1+ntypes_s) * nhist[s]
 * values, total first), pair sums at rows type_first[s] .. of S.
 * totals = {hist_len, pdf_len, ntypes_total}.  Any output may be NULL. */
int xs_batch_info(const xs_batch *plan, unsigned *nhist,
                  unsigned long long *hist_off, unsigned long long *pdf_off,
                  unsigned long long *type_first, unsigned long long *totals);

/* Histograms of every structure (as xs_hist), then, if S != NULL and nq > 0,
 * pair sums S[t*nq+iq] of every pair type t (as xs_hist_pairsum, one q mesh
 * for all; bin by bin where the memory for the node tables cannot be had),
 * then, if pdf != NULL, PDFs of pdf_type (as xs_pdf) with rho0[s]
 * and sl[] in el_count order.  XS_DEVICE_PTRS: hist, q, S and pdf are device
 * pointers and the call returns without waiting; else host arrays and the
 * call is synchronous.  XS_BATCH_GRAPH: the launches are captured into a
 * hipGraph on the first call and replayed by later calls with the same
 * pointers, nq, pdf_type and flags (needs a non-default stream).
 * XS_PAIRSUM_MFMA: the pair sums as int8 matrix-core products (as
 * xs_hist_pairsum with that flag), with the pair types grouped by bin count
 * and count slices taken from each type's pair count (no read-back, so the
 * run stays capturable); XS_ERR_RANGE if a pair type has 2^35 pairs or more.
 * Its error is absolute, at most 2^-35 x (sum of the type's counts) per S
 * entry, so relative to I(q) it grows with the structure's atom count.
 * Its slices take about 5*nq*max(nhist) + (count slices)*sum(nhist) bytes of
 * the plan's run buffer.
 * Overlapping runs of one plan race; use one plan per stream. */
int xs_batch_run(xs_batch *plan, uint64_t *hist, const double *q, unsigned nq,
                 double *S, int pdf_type, const double *rho0, const double *sl,
                 double *pdf, unsigned flags);

/* Per-structure overflow counts of the last run (host array, synchronous). */
int xs_batch_overflow(xs_batch *plan, uint64_t *overflow);

/* Free a plan.  xs_free frees the plans of its context that are still
 * alive; a plan must not be used or freed after its context is freed. */
int xs_batch_free(xs_batch *plan);

/* Ensemble builder.  One structural block as block::calcAtoms receives it
 * after ReadConfig (ReadXML.cpp:254-323): cell atoms made absolute
 * (redefAtoms, CalcFunctions.cpp:116-127) and sorted element-major
 * (block::sortAtoms, 158-196), symmetry translations made absolute
 * (redefSymm, 128-133), copies' rotation rows from calcRotMatrix.
 * 3-vectors are row-major: r_atom[a*3+k]; p_symm[s*9 + row*3 + col] holds
 * rows R1, R2, R3 of SymmEqPos s (s = 0 is the identity); cell = a, b, c;
 * cf[c*9 + row*3 + col] the rotation rows of copy c.  el[a] is the ensemble
 * element of cell atom a (block::id of its type).  rcut > 0 keeps atoms with
 * |r - r_mean|^2 <= rcut^2 (CutOff Rcut), rcut_copies > 0 those within
 * rcut_copies of the mean copy position (CutOff RcutCopies); dev[a] and
 * dev_mol are standard deviations (sqrt of Uiso, mol_Uiso). */
typedef struct xs_block_desc {
  unsigned natom, nsymm, ncopy;
  unsigned ncell[3];
  const unsigned *el;
  const double *r_atom, *occ, *dev, *p_symm, *r_symm, *cell, *r_copy, *cf;
  double r_mean[3];
  double rcut, rcut_copies, dev_mol;
  int mol_rotation;
} xs_block_desc;

/* Build the atoms of an ensemble of blocks on the device.  Replaces
 * CalcAndPrintAtoms' loop over block::calcAtoms (CalcFunctions.cpp:398-404,
 * 251-397): symmetry images of the cell atoms; images closer than 0.5 A
 * under translations of up to +-2 cells share one position and their
 * occupancies add up across elements; then, for every copy and cell, one
 * occupancy draw per covering site places at most one atom, with the atom
 * and molecule displacements, molecule rotations and cut-offs of the
 * reference.  Positions are computed in FP64 with the reference's operation
 * order, so without random terms they equal its atoms bit for bit.  The
 * clock-seeded default_random_engine of the reference is replaced by
 * Philox4x64-10 counters keyed by (seed, block), so one seed gives one
 * ensemble whatever the launch order.  Blocks' descriptions are host memory
 * and are not kept.  The result stays on the device until xs_atoms_free. */
int xs_atoms_build(xs_ctx *ctx, const xs_block_desc *blocks, unsigned nblocks, unsigned n_el,
                   uint64_t seed, xs_atoms **atoms);

/* Counts of the built ensemble: el_count[n_el] (NatomEl of
 * CalcAndPrintAtoms, 405-408), block_el_count[nblocks*n_el] (NatomElAll of
 * each block), *n_atoms (Ntot).  Any output may be NULL. */
int xs_atoms_info(const xs_atoms *atoms, unsigned *el_count, unsigned *block_el_count,
                  uint64_t *n_atoms);

/* Copy the atoms as element-major SoA xyz[3*n_atoms] (within an element:
 * block, copy, cell, site order -- the order of the reference's ra[el]).
 * XS_DEVICE_PTRS: xyz is device memory (enqueued on the context stream),
 * else host memory (synchronous). */
int xs_atoms_copy(xs_atoms *atoms, double *xyz, unsigned flags);

/* Free a built ensemble.  xs_free frees those of its context still alive. */
int xs_atoms_free(xs_atoms *atoms);

#ifdef __cplusplus
}
#endif
#endif /* XS_HIP_H */
