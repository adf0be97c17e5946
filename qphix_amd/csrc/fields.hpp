// Host-side declarations shared by the library translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include "common.hpp"
#include <stdint.h>

namespace qphix_amd {

// lattice + precision descriptor of a geometry
struct GeomDesc {
  int L[4];
  int prec;   // Prec
  int c12;    // two-row gauge compression
  long vh;    // sites per checkerboard
  size_t vs;  // plane stride in sites
};

hipError_t fld_pack_spinor(const GeomDesc &g, void *dst, const double *dsrc, hipStream_t st);
hipError_t fld_unpack_spinor(const GeomDesc &g, double *ddst, const void *src, hipStream_t st);
hipError_t fld_gen_spinor(const GeomDesc &g, void *dst, uint64_t seed, int cb, hipStream_t st);
hipError_t fld_convert_spinor(const GeomDesc &go, void *out, double scale, const GeomDesc &gi, const void *in,
                              hipStream_t st);
hipError_t fld_pack_gauge_cb(const GeomDesc &g, void *dst, int cb, const double *dsrc, hipStream_t st);
hipError_t fld_gen_gauge_canonical(const GeomDesc &g, double *du, uint64_t seed, double eps, hipStream_t st);
hipError_t fld_convert_gauge(const GeomDesc &go, void *out, const GeomDesc &gi, const void *in, hipStream_t st);
hipError_t fld_pack_clover(const GeomDesc &g, void *dst, const double *dsrc, hipStream_t st);
hipError_t fld_unpack_clover(const GeomDesc &g, double *ddst, const void *src, hipStream_t st);
hipError_t fld_pack_full_clover(const GeomDesc &g, void *dst, const double *dsrc, hipStream_t st);
hipError_t fld_convert_clover(const GeomDesc &go, void *out, const GeomDesc &gi, const void *in, int full,
                              hipStream_t st);
hipError_t fld_clover_build(const GeomDesc &g, const void *u0, const void *u1, double cr, double ct, double dm,
                            int cb, int what, double mu, double eps, void *out, hipStream_t st);

// BLAS operations (one spinor per operand; see blas.hip)
enum BlasOp {
  B_COPY = 0, B_ZERO, B_AXY, B_AX, B_YPEQX, B_YMEQX, B_AYPX, B_AXPY, B_AXPBY,
  B_NORM2, B_AXPYNORM2, B_XMYNORM2, B_XMY2NORM2, B_RMAMMP, B_RICH, B_BICG_XMY,
  B_CDOT, B_CDOTNORM, B_PUPD, B_SUPD, B_CAXPY, B_RXUPD, B_MRUPD, B_TWM, B_TWM2,
  B_CLOVMULT, B_FULLMULT, B_TWOFLAV_INVCLOV, B_RXUPD_CDOT, NUM_BLAS_OPS
};
struct BlasArgs {
  const void *x, *y, *z, *w;  // read-only operands
  void *o0, *o1, *o2, *o3;    // written (and possibly read) operands
  double a[6];                // scalars
  // non-null: the scalars are read from device memory, dsc[0..5], when the
  // kernel starts, and the launch does nothing if dsc[7] != 0 (a solver
  // whose device state says it is done)
  const double *dsc;
};
int blas_nred(int op);
// What the last work-group of a reduction does with the sums: it writes them
// to out (device or pinned host memory) and takes the scalar step of a
// device-resident solver loop on `state` (the sums being fields of it)
enum BlasTail { TAIL_NONE = 0, TAIL_CG_MID, TAIL_CG_POST, TAIL_BI_MID, TAIL_BI_MID2, TAIL_BI_POST, TAIL_MS_MID, TAIL_MS_POST };
struct BlasFin {
  double *partials;  // per work-group sums, kMaxBlasBlocks * 3 doubles
  unsigned *tickets;  // kTickets counters of work-groups done, 0 between launches;
                      // not shared with a launch that may overlap this one
  double *out;
  int tail;
  void *state;
};
// launches op over the geometry; reductions end in fin (BlasFin), without a
// further launch
hipError_t blas_launch(const GeomDesc &g, int op, const BlasArgs &a, const BlasFin &fin, hipStream_t st);
constexpr int kMaxBlasBlocks = 2048;
constexpr int kTicketGroup = 64, kTicketStride = 32;  // work-groups per counter, a counter per 128 bytes
constexpr int kTickets = (1 + kMaxBlasBlocks / kTicketGroup) * kTicketStride;
// a kernel, so that it may be captured
hipError_t blas_clear_tickets(unsigned *tickets, hipStream_t st);

// Multishift CG vector updates for every shift in one sweep (minvcg.h:298-363):
//   x_s -= beta_s p_s      for s in mask_x   (uses p_s before its update)
//   p0   = r + a p0        if do_p0
//   p_s  = zeta_s r + as_s p_s   for s in mask_p
constexpr int kMaxShifts = 32;
struct MShiftArgs {
  const void *r;
  void *p0;
  void *p[kMaxShifts];
  void *x[kMaxShifts];
  double a;
  double zeta[kMaxShifts], as[kMaxShifts], beta[kMaxShifts];
  unsigned mask_x, mask_p;
  int do_p0, nshift;
};
hipError_t mshift_launch(const GeomDesc &g, const MShiftArgs &m, hipStream_t st);

// What a device-resident solver loop publishes at the end of every iteration
// into view[posts & 1] of a pinned host array: the host reads the state of a
// finished iteration without a copy command (progress: the residual over its
// target, below 1 once converged)
struct SolverView {
  int done, pad;
  double progress;
};

// One iteration's vector updates of the shifted systems, in order:
// x_s -= beta_s p_s (mask_x), then p_s = zeta_s r + as_s p_s (mask_p)
struct MsRec {
  double beta[kMaxShifts], zeta[kMaxShifts], as[kMaxShifts];
  unsigned mask_x, mask_p;
};
// Iterations whose updates of the shifted systems are applied in one sweep
constexpr int kMsDepth = 8;
// Multishift CG state in device memory (minvcg.h:279-384): the FP64 scalars
// and per-shift recurrences of one solve, updated where the reductions end
// (BlasTail), so that an iteration needs no host round trip and can be
// captured in a HIP graph. cf[f] receives per-flavour reductions. Iteration k
// keeps its updates in rec[k % depth].
struct MsState {
  double b, bp, c, cp, d;
  double p0upd[8];  // the p0 update's scalars (BlasArgs::dsc): a, and the skip flag
  double cf[2];
  double shifts[kMaxShifts], zeta[kMaxShifts], zeta_prev[kMaxShifts], beta[kMaxShifts];
  double rsd_sq[kMaxShifts], rsd_sq_final[kMaxShifts];
  int conv[kMaxShifts];
  int nshift, nf, iters, max_iters, done, converged;
  int depth, at;  // at: the record of the next sweep
  unsigned long site_flops;
  // largest c zeta_s^2 / target_s over the shifts tested by the last
  // iteration (below 1 for a shift that converged there); lets the host
  // foresee the last iteration
  double progress;
  SolverView *hview;
  int posts, pad;
  MsRec *rec;  // kMsDepth records, right after the state
};
// the recorded updates of all shifts (m.p, m.x) in one sweep over r[0 .. depth - 1]
// and, with do_p0, p0 = r[0] + a p0 (depth 1 only)
struct MsSweep {
  const void *r[kMsDepth];
  void *p0;
  void *p[kMaxShifts];
  void *x[kMaxShifts];
  int nshift, depth;
};
hipError_t ms_sweep_launch(const GeomDesc &g, const MsSweep &m, const MsState *st_dev, hipStream_t st);
// start of the first iteration: a = c / cp, as_s, mask_p, cp = c, bp = b
hipError_t ms_pre_launch(MsState *st_dev, hipStream_t st);
// TAIL_MS_MID: b = -cp / d, d the sum of cf over flavours.
// TAIL_MS_POST: end of an iteration, c from cf, zeta / beta recurrences,
// convergence, then the start of the next iteration as ms_pre_launch (or, once
// the solve is done, only the pending x_s updates for the next sweep)
// BiCGStab state in device memory (invbicgstab.h:150-256): the complex
// scalars, the reductions the device loop writes (<r0, v>, <t, r> with |t|^2,
// |r|^2 with <r0, r>), and the scalar blocks of the three vector updates
// (BlasArgs::dsc; [7] = skip once done). Updated where the reductions end
// (BlasTail), so one iteration needs no host round trip.
struct BiState {
  double rho[2], rho_prev[2], alpha[2], omega[2];
  double r0v[2], tr[3], ru[3];
  double r_norm, rsd_sq;
  double pupd[8], supd[8], rxupd[8];
  unsigned long site_flops, mv_apps, sf;  // sf: the reference's unit, 12 x flavours
  int iters, max_iters, done, status, n_iters, posts;
  double progress;
  SolverView *hview;
};
// start of the first iteration: rho = <r0, r>, the breakdown test, beta,
// p-update scalars. The tails: TAIL_BI_MID after v = M p and <r0, v>, the
// breakdown test, alpha, s-update scalars; TAIL_BI_MID2 after t = M r, <t, r>
// and |t|^2, the breakdown test, omega, x/r-update scalars; TAIL_BI_POST after
// the x/r update, |r|^2, convergence, the iteration count and the start of the
// next iteration
hipError_t bi_pre_launch(BiState *st_dev, hipStream_t st);
// *st_dev = h
hipError_t bi_set_launch(BiState *st_dev, const BiState &h, hipStream_t st);

// CG state in device memory (invcg.h:88-456): c = |r|^2 of the iteration,
// the reductions |M p|^2 and |r|^2, the scalar blocks of the two vector
// updates (BlasArgs::dsc; [7] = skip once done), the counters
struct CgDState {
  double c, d_raw, r_raw, rsd_sq, cp;
  double rmammp[8], aypx[8];
  unsigned long site_flops, mv_apps, sf;
  int iters, max_iters, done, status, n_iters, posts;
  double rsd_sq_final, progress;
  SolverView *hview;
};
// TAIL_CG_MID after M^+M p and |M p|^2: a = c / d. TAIL_CG_POST after
// r -= a M^+M p, x += a p, |r|^2: convergence, b = |r|^2 / c
hipError_t cgd_set_launch(CgDState *st_dev, const CgDState &h, hipStream_t st);
hipError_t ms_set_launch(MsState *st_dev, const MsState &h, hipStream_t st);

// o = y + (*b) x and |o|^2, the scalar read from device memory (o may be y)
hipError_t axpy_norm2_dev_launch(const GeomDesc &g, const double *b, const void *x, const void *y, void *o,
                                 const BlasFin &fin, hipStream_t st);

// one BLAS operation on n right-hand sides in one launch, each with its own
// operands and first scalar; reductions come back per right-hand side
struct MultiBlasArgs {
  const void *x[kMaxRhs];
  const void *y[kMaxRhs];
  void *o0[kMaxRhs];
  void *o1[kMaxRhs];
  double a[kMaxRhs];
  int n;
};
// partials must hold kMaxBlasBlocks * 3 doubles; out n * nred doubles
hipError_t blas_multi_launch(const GeomDesc &g, int op, const MultiBlasArgs &m, double *partials, double *out,
                             hipStream_t st);

// streaming calibration kernel (words per site in / out: 30, 48, 60, 66 / 6; 120 / 12)
hipError_t stream_launch(const GeomDesc &g, int nwi, int nwo, const void *in, void *out, hipStream_t st);

// records msg as the thread's last error (qphix_last_error) and returns code
int api_fail(int code, const char *msg);

}  // namespace qphix_amd
