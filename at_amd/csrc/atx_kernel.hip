// atx_kernel.hip -- persistent FP64 tracking kernel for gfx950 (MI355X).
//
// One lane tracks one particle through every element of every turn in a
// single launch; the particle's 6-vector lives in registers from the first
// load to the final store, and HBM is touched only at start, at refpt
// copies, on a loss and at the end. A lattice is a list of records (LatOp,
// prepared by atx_host.cpp) read through the constant address space: every
// lane of a wave is at the same record, so its constants land in SGPRs and
// its branches are scalar. The loop over the records has no divergent branch
// (losses, the only ones, are handled in a function that the whole wave
// calls), and keeps the common elements inline and all others in functions;
// lattices with rarer forms or maps (OPF_FULL) take a loop that has those, too.
//
// This file is compiled twice:
//   ATX_STRICT=1, -ffp-contract=off: the reference operation order of
//     atintegrators/*.c, with the same divisions, so results agree bit for
//     bit with the CPU reference except where a device transcendental (sin in
//     RFCavityPass, tan in per-particle edge fringes) enters;
//   ATX_STRICT=0, -ffp-contract=on: the same maps with FMA contraction,
//     hand-fused Horner steps and the 1/(1+delta) reciprocals hoisted where
//     delta is constant; agreement with the reference is to rounding.
#include <hip/hip_runtime.h>

#include <limits.h>

#include "atx_device.h"
#include "atx_libm.h"

#ifndef ATX_STRICT
#error "ATX_STRICT must be defined to 0 or 1"
#endif
// One object per launch shape (particles per lane ATX_PPT, slices per loop
// iteration ATX_UNROLL) and build, compiled in parallel; the helper kernels
// (repack, live map, diffusion matrices) go into the strict 1x1 object.
#if !defined(ATX_PPT) || !defined(ATX_UNROLL)
#error "ATX_PPT (1, 2) and ATX_UNROLL (1, 2, 4) must be defined"
#endif
#define ATX_AUX (ATX_STRICT && ATX_PPT == 1 && ATX_UNROLL == 1)
#define ATX_PASTE6(a, b, c, d, e, f) a##b##c##d##e##f
#define ATX_NAME(build, p, u) ATX_PASTE6(atx_launch_track_, build, _p, p, _u, u)

#if ATX_STRICT
#define ATX_NS strict_ns
#define ATX_LAUNCH ATX_NAME(strict, ATX_PPT, ATX_UNROLL)
#else
#define ATX_NS fast_ns
#define ATX_LAUNCH ATX_NAME(fast, ATX_PPT, ATX_UNROLL)
#endif

namespace atx {
namespace ATX_NS {

// Read-only element data: constant address space -> scalar loads.
typedef __attribute__((address_space(4))) const double cdouble;
typedef __attribute__((address_space(4))) const DevElem cDevElem;
typedef __attribute__((address_space(4))) const Instance cInstance;
typedef __attribute__((address_space(4))) const LatOp cLatOp;
typedef __attribute__((address_space(4))) const int32_t cint;

struct R6 {
  double x, px, y, py, dp, ct;
};

// Forest-Ruth 4th-order coefficients (atintegrators/atconstants.h:15-19);
// only their products with the slice length are used, prepared on the host.

__device__ __forceinline__ void add_t(R6& r, cdouble* t) {
  r.x += t[0];
  r.px += t[1];
  r.y += t[2];
  r.py += t[3];
  r.dp += t[4];
  r.ct += t[5];
}

// Per-element (not per-slice) maps that are large or use transcendentals are
// kept out of line: inlined into every element variant they would multiply
// the kernel's code size and register demand (a 6x6 matrix alone holds 72
// SGPRs), while they run at most a few times per element.

// r <- M r with M column-major (atlalib.c:17-32); the sum starts from 0.0 as
// in the reference.
__device__ __forceinline__ R6 mul_r_inl(const R6& r, cdouble* m) {
  const double v[6] = {r.x, r.px, r.y, r.py, r.dp, r.ct};
  double o[6];
#pragma unroll
  for (int i = 0; i < 6; i++) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < 6; j++) s += m[i + 6 * j] * v[j];
    o[i] = s;
  }
  return R6{o[0], o[1], o[2], o[3], o[4], o[5]};
}

__device__ __noinline__ R6 mul_r_v(R6 r, cdouble* m) { return mul_r_inl(r, m); }

__device__ __forceinline__ void mul_r(R6& r, cdouble* m) { r = mul_r_v(r, m); }

// atlalib.c:70-75
__device__ __noinline__ R6 change_pref_v(R6 r, double s) {
  r.px /= s;
  r.py /= s;
  r.dp = (r.dp + 1.0 - s) / s;
  return r;
}

__device__ __forceinline__ void change_pref(R6& r, double s) { r = change_pref_v(r, s); }

// Apertures are decisions: evaluated without contraction in both builds so
// that the loss element is the reference's (atlalib.c:164-190).
template <class L>
__device__ __forceinline__ void rect_ap(R6& r, const L& lim) {
#pragma clang fp contract(off)
  const bool out = (r.x < lim[0]) | (r.x > lim[1]) | (r.y < lim[2]) | (r.y > lim[3]);
  r.ct = out ? __builtin_inf() : r.ct;
}

__device__ __forceinline__ void ellip_ap(R6& r, cdouble* ax) {
#pragma clang fp contract(off)
  const double u = r.x / ax[0];
  const double v = r.y / ax[1];
  if ((u * u + v * v) >= 1.0) r.ct = __builtin_inf();
}

__device__ __forceinline__ void apertures(R6& r, cDevElem& h, cdouble* pool) {
  if (h.flags & F_RAP) rect_ap(r, pool + h.rap);
  if (h.flags & F_EAP) ellip_ap(r, pool + h.eap);
}

__device__ __forceinline__ void entry_xform(R6& r, cDevElem& h, cdouble* pool) {
  if (h.flags & F_T1) add_t(r, pool + h.t1);
  if (h.flags & F_R1) mul_r(r, pool + h.r1);
}

__device__ __forceinline__ void exit_xform(R6& r, cDevElem& h, cdouble* pool) {
  if (h.flags & F_R2) mul_r(r, pool + h.r2);
  if (h.flags & F_T2) add_t(r, pool + h.t2);
}

#if !ATX_STRICT
// Fast build: 1/d from the hardware reciprocal estimate (v_rcp_f64) and two
// Newton steps q <- q + q (1 - d q), each of which squares the relative
// error of the estimate; the result is within an ulp of 1/d.
__device__ __forceinline__ double fast_rcp(double d) {
  double q = __builtin_amdgcn_rcp(d);
  double e = __builtin_fma(-d, q, 1.0);
  q = __builtin_fma(q, e, q);
  e = __builtin_fma(-d, q, 1.0);
  return __builtin_fma(q, e, q);
}
#endif

// Full drift with its own 1/(1+delta) (atlalib.c:59-68, driftkickrad.c:36-45,
// diff_drift.c:30-43 share this arithmetic); the fast build takes fast_rcp
// for the division.
__device__ __forceinline__ void drift6(R6& r, double len) {
#if ATX_STRICT
  const double pn = 1.0 / (1.0 + r.dp);
#else
  const double pn = fast_rcp(1.0 + r.dp);
#endif
  const double nl = len * pn;
  r.x += nl * r.px;
  r.y += nl * r.py;
  r.ct += nl * pn * (r.px * r.px + r.py * r.py) / 2.0;
}

// In-magnet drift with nl = L/(1+delta) hoisted (driftkick.c:37-48).
// h2 = 1/(2(1+delta)) is used by the fast build only.
__device__ __forceinline__ void fastdrift(R6& r, double nl, double h2) {
#if ATX_STRICT
  (void)h2;
  r.x += nl * r.px;
  r.y += nl * r.py;
  r.ct += nl * (r.px * r.px + r.py * r.py) / (2.0 * (1.0 + r.dp));
#else
  r.x = __builtin_fma(nl, r.px, r.x);
  r.y = __builtin_fma(nl, r.py, r.y);
  const double p2 = __builtin_fma(r.px, r.px, r.py * r.py);
  r.ct = __builtin_fma(nl * p2, h2, r.ct);
#endif
}

// Addends of the first Horner step, B[order-1] and A[order-1] (0 for order
// 0), taken once per magnet. That step multiplies the constants B[order],
// A[order] by a coordinate and adds another constant, and an FMA reads at
// most one SGPR: the fast build therefore keeps these two addends in VGPRs
// for the whole magnet instead of moving them from SGPRs at every kick.
template <int N>
__device__ __forceinline__ void horner_addends(cdouble* a, cdouble* b, int n, double& blo,
                                               double& alo) {
  const int order = (N >= 0) ? N : n;
  blo = (order >= 1) ? b[order - 1] : 0.0;
  alo = (order >= 1) ? a[order - 1] : 0.0;
#if !ATX_STRICT
  if (N >= 1) {
    asm("" : "=v"(blo) : "0"(blo));
    asm("" : "=v"(alo) : "0"(alo));
  }
#endif
}

// Horner evaluation of sum (B_k + i A_k)(x + i y)^k (driftkick.c:92-110).
// N >= 0: order known at compile time; N < 0: runtime order n. blo, alo:
// B[order-1], A[order-1] from horner_addends (the same values).
template <int N>
__device__ __forceinline__ void field(const R6& r, cdouble* a, cdouble* b, int n, double blo,
                                      double alo, double& re, double& im) {
  const int order = (N >= 0) ? N : n;
  re = b[order];
  im = a[order];
#pragma unroll
  for (int k = order - 1; k >= 0; k--) {
    const double bk = (N >= 1 && k == order - 1) ? blo : b[k];
    const double ak = (N >= 1 && k == order - 1) ? alo : a[k];
#if ATX_STRICT
    const double t = re * r.x - im * r.y + bk;
    im = im * r.x + re * r.y + ak;
#else
    const double t = __builtin_fma(re, r.x, __builtin_fma(-im, r.y, bk));
    im = __builtin_fma(im, r.x, __builtin_fma(re, r.y, ak));
#endif
    re = t;
  }
}

// driftkick.c:92-115
template <int N>
__device__ __forceinline__ void str_kick(R6& r, cdouble* a, cdouble* b, int n, double blo,
                                         double alo, double kl) {
  double re, im;
  field<N>(r, a, b, n, blo, alo, re, im);
  r.px -= kl * re;
  r.py += kl * im;
}

// driftkick.c:51-89; kli = kl*irho prepared on the host
template <int N>
__device__ __forceinline__ void bnd_kick(R6& r, cdouble* a, cdouble* b, int n, double blo,
                                         double alo, double kl, double irho, double kli) {
  double re, im;
  field<N>(r, a, b, n, blo, alo, re, im);
#if ATX_STRICT
  r.px -= kl * (re - (r.dp - r.x * irho) * irho);
  r.py += kl * im;
  r.ct += kli * r.x;
#else
  const double u = __builtin_fma(-r.x, irho, r.dp);
  const double v = __builtin_fma(-u, irho, re);
  r.px = __builtin_fma(-kl, v, r.px);
  r.py = __builtin_fma(kl, im, r.py);
  r.ct = __builtin_fma(kli, r.x, r.ct);
#endif
}

// Radiating drift (diff_drift.c:30-43).
__device__ __forceinline__ void rad_drift(R6& r, double len, double pn) {
  const double nl = len * pn;
  r.x += nl * r.px;
  r.y += nl * r.py;
  r.ct += nl * pn * (r.px * r.px + r.py * r.py) / 2.0;
}

#if !ATX_STRICT
// One Newton step: for a reciprocal that only scales the radiated energy (a
// relative change of 1e-8 or less per kick), where an error of the squared
// estimate error is far below the rounding of delta.
__device__ __forceinline__ double rcp1(double d) {
  const double q = __builtin_amdgcn_rcp(d);
  return __builtin_fma(q, __builtin_fma(-d, q, 1.0), q);
}

// Fast build: reciprocal of 1 + delta after a kick from the one before it,
// pn = 1/(1 + delta_before). With the radiated fraction e = 1 - (1 + delta) pn
// (about 1e-7 per kick), 1/(1 + delta) = pn/(1 - e) = pn (1 + e + e^2) to a
// relative e^3, below 1e-17 for |e| <= 2e-6. A wave in which any lane
// radiated more than that in one kick takes fast_rcp.
__device__ __forceinline__ double rcp_after_kick(double opd2, double pn) {
  const double e = __builtin_fma(-opd2, pn, 1.0);
  double q = __builtin_fma(pn, __builtin_fma(e, e, e), pn);
  const bool far = __builtin_fabs(e) > 2e-6;
  // a select under the vote: no divergent branch in the slices
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(far) != 0, 0)) q = far ? fast_rcp(opd2) : q;
  return q;
}
#endif

// Radiating straight kick (diff_str_kick.c:19-83, bdiff == NULL).
// radc = RAD_CONST*gamma^3 (strict); radk = radc*kl (fast). Takes pn =
// 1/(1+delta) at entry and returns it for the radiated delta.
template <int N>
__device__ __forceinline__ void rad_str_kick(R6& r, cdouble* a, cdouble* b, int n, double blo,
                                             double alo, double kl, double radc, double radk,
                                             double& pn_io) {
  double re, im;
  field<N>(r, a, b, n, blo, alo, re, im);
#if ATX_STRICT
  (void)radk;
  double pn = pn_io;
  const double xpr = r.px * pn;
  const double ypr = r.py * pn;
  const double vn2 = 1.0 / (1.0 + xpr * xpr + ypr * ypr);
  const double cr = im * ypr - re * xpr;
  const double b2p = (re * re + im * im + cr * cr) * vn2;
  const double factor = (1.0 + (xpr * xpr + ypr * ypr) / 2.0) / (pn * pn) * kl;
  r.dp -= radc * b2p * factor;
  pn = 1.0 / (1.0 + r.dp);
  r.px = xpr / pn;
  r.py = ypr / pn;
  r.px -= kl * re;
  r.py += kl * im;
  pn_io = pn;
#else
  (void)radc;
  const double pn_in = pn_io;
  const double opd = 1.0 + r.dp;
  const double xpr = r.px * pn_in;
  const double ypr = r.py * pn_in;
  const double s2 = __builtin_fma(xpr, xpr, ypr * ypr);
  const double cr = __builtin_fma(im, ypr, -re * xpr);
  const double b2 = __builtin_fma(cr, cr, __builtin_fma(re, re, im * im));
  // g = (1+s2/2)/(1+s2) = 1 - (s2/2)/(1+s2), with 1 - s2 + s2^2 for the
  // reciprocal: relative error s2^4/2 in g, below 1e-16 for s2 <= 1e-4
  // (angles up to 10 mrad); a wave with a wider angle divides.
  double g = __builtin_fma(-0.5 * s2, __builtin_fma(s2, s2, 1.0 - s2), 1.0);
  const bool wide = s2 > 1e-4;
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(wide) != 0, 0))
    g = wide ? __builtin_fma(0.5, s2, 1.0) * rcp1(1.0 + s2) : g;
  r.dp = __builtin_fma(-radk, (b2 * g) * (opd * opd), r.dp);
  const double opd2 = 1.0 + r.dp;
  r.px = __builtin_fma(xpr, opd2, -kl * re);
  r.py = __builtin_fma(ypr, opd2, kl * im);
  pn_io = rcp_after_kick(opd2, pn_in);
#endif
}

// Radiating curved-frame kick (diff_bnd_kick.c:85-174, bdiff == NULL).
template <int N>
__device__ __forceinline__ void rad_bnd_kick(R6& r, cdouble* a, cdouble* b, int n, double blo,
                                             double alo, double kl, double irho, double kli,
                                             double radc, double radk, double& pn_io) {
  double re, im;
  field<N>(r, a, b, n, blo, alo, re, im);
#if ATX_STRICT
  (void)radk;
  double pn = pn_io;
  const double x = r.x;
  const double xpr = r.px * pn;
  const double ypr = r.py * pn;
  const double by = re + irho;
  const double bx = im;
  const double hx = 1.0 + x * irho;
  const double vn2 = 1.0 / (hx * hx + xpr * xpr + ypr * ypr);
  const double byh = by * hx;
  const double bxh = bx * hx;
  const double cr = bx * ypr - by * xpr;
  const double b2p = (byh * byh + bxh * bxh + cr * cr) * vn2;
  const double factor = (1.0 + x * irho + (xpr * xpr + ypr * ypr) / 2.0) / (pn * pn) * kl;
  const double d0 = r.dp;
  r.dp -= radc * b2p * factor;
  pn = 1.0 / (1.0 + r.dp);
  r.px = xpr / pn;
  r.py = ypr / pn;
  r.px -= kl * (re - (d0 - r.x * irho) * irho);
  r.py += kl * im;
  r.ct += kli * r.x;
  pn_io = pn;
#else
  (void)radc;
  const double pn_in = pn_io;
  const double x = r.x;
  const double opd = 1.0 + r.dp;
  const double xpr = r.px * pn_in;
  const double ypr = r.py * pn_in;
  const double by = re + irho;
  const double hx = __builtin_fma(x, irho, 1.0);
  const double s2 = __builtin_fma(xpr, xpr, ypr * ypr);
  const double byh = by * hx;
  const double bxh = im * hx;
  const double cr = __builtin_fma(im, ypr, -by * xpr);
  const double b2 = __builtin_fma(cr, cr, __builtin_fma(byh, byh, bxh * bxh));
  const double g = __builtin_fma(0.5, s2, hx) * rcp1(__builtin_fma(hx, hx, s2));
  const double d0 = r.dp;
  r.dp = __builtin_fma(-radk, (b2 * g) * (opd * opd), r.dp);
  const double opd2 = 1.0 + r.dp;
  const double u = __builtin_fma(-x, irho, d0);
  const double v = __builtin_fma(-u, irho, re);
  r.px = __builtin_fma(xpr, opd2, -kl * v);
  r.py = __builtin_fma(ypr, opd2, kl * im);
  r.ct = __builtin_fma(kli, x, r.ct);
  pn_io = rcp_after_kick(opd2, pn_in);
#endif
}

// Edge focusing (atphyslib.c:15-79, diff_bend_fringe.c:2-53). sgn = +1 at
// the entrance, -1 at the exit; fx, c0 = irho*tan(edge), edge and corr/psi
// come from the scalar block.
__device__ __noinline__ double edge_fy_tan(int mode, double dp, double px, double irho,
                                           double edge_angle, double corr, double sgn) {
  switch (mode) {
    case E_TAN1:
      return irho * tan(edge_angle - corr / (1.0 + dp));
    case E_TAN2:
      return irho * tan(edge_angle - corr / (1.0 + dp)) / (1.0 + dp);
    case E_TAN3:
      return (sgn > 0.0) ? irho * tan(edge_angle - corr + px / (1.0 + dp))
                         : irho * tan(edge_angle - corr - px / (1.0 + dp));
    case E_RTAN1: {
      const double pn = 1.0 / (1.0 + dp);
      return irho * tan(edge_angle - corr * pn);
    }
    case E_RTAN2: {
      const double pn = 1.0 / (1.0 + dp);
      return irho * tan(edge_angle - corr * pn) * pn;
    }
    default: {  // E_RTAN3
      const double pn = 1.0 / (1.0 + dp);
      return irho * tan(edge_angle - corr + sgn * px * pn);
    }
  }
}

template <bool LEAN>
__device__ __forceinline__ void edge(R6& r, int mode, double irho, double fx, double c0,
                                     double edge_angle, double corr, double sgn) {
  double fy;
  if (mode == E_CONST)
    fy = c0;
  else if (mode == E_DIVP)
    fy = c0 / (1.0 + r.dp);
  else if (LEAN || mode == E_MULPN)
    fy = c0 * (1.0 / (1.0 + r.dp));
  else
    fy = edge_fy_tan(mode, r.dp, r.px, irho, edge_angle, corr, sgn);
  r.px += r.x * fx;
  r.py -= r.y * fy;
}

// Lee-Whiting hard-edge quadrupole fringe (quadfringe.c:3-51).
__device__ __forceinline__ void quad_fringe_inl(R6& r, double b2, bool entrance) {
  const double u = b2 / (12.0 * (1.0 + r.dp));
  const double x2 = r.x * r.x;
  const double z2 = r.y * r.y;
  const double xz = r.x * r.y;
  const double gx = u * (x2 + 3.0 * z2) * r.x;
  const double gz = u * (z2 + 3.0 * x2) * r.y;
  const double dpx = 3.0 * u * (2.0 * xz * r.py - (x2 + z2) * r.px);
  const double dpy = 3.0 * u * (2.0 * xz * r.px - (x2 + z2) * r.py);
  if (entrance) {
    r.x += gx;
    r.y -= gz;
    r.ct -= (gz * r.py - gx * r.px) / (1.0 + r.dp);
    r.px += dpx;
    r.py -= dpy;
  } else {
    r.x -= gx;
    r.y += gz;
    r.ct += (gz * r.py - gx * r.px) / (1.0 + r.dp);
    r.px -= dpx;
    r.py += dpy;
  }
}

// 2x2 linear blocks of the elegant fringe (quadfringe.c:93-163), matrices
// prepared on the host: m = {Rxx, Rxp, Rpx, Rpp, Ryy, Ryq, Rqy, Rqq}.
__device__ __forceinline__ void apply_2x2(R6& r, cdouble* m) {
  const double x = r.x, px = r.px, y = r.y, py = r.py;
  r.x = m[0] * x + m[1] * px;
  r.px = m[2] * x + m[3] * px;
  r.y = m[4] * y + m[5] * py;
  r.py = m[6] * y + m[7] * py;
}

// mode: Q_LEE or Q_ELEGANT; m: the two 2x2 blocks around the Lee-Whiting map
__device__ __noinline__ R6 quad_fringe_v(R6 r, int mode, cdouble* m, double b2, bool entrance) {
  if (mode == Q_ELEGANT) apply_2x2(r, m);
  quad_fringe_inl(r, b2, entrance);
  if (mode == Q_ELEGANT) apply_2x2(r, m + 8);
  return r;
}

__device__ __forceinline__ void quad_fringe_in(R6& r, cDevElem& h, cdouble* pool, double b2) {
  r = quad_fringe_v(r, h.fringe & 0xff, pool + h.fq, b2, true);
}

__device__ __forceinline__ void quad_fringe_out(R6& r, cDevElem& h, cdouble* pool, double b2) {
  r = quad_fringe_v(r, (h.fringe >> 8) & 0xff, pool + h.fq + 16, b2, false);
}

// Slices of a non-default integrator (atgpu/SymplecticIntegrator.cpp types
// 1-3, 5, 6): the host-built op table lists the drifts and kicks of one
// slice; kept out of line, generic in the multipole order.
template <bool BEND, bool RAD>
__device__ __noinline__ R6 slices_ops(R6 r, cdouble* a, cdouble* b, int n, cdouble* op, int nslice,
                                      double pn0, double irho, double radc) {
  const int nop = (int)op[0];
  double blo, alo;
  horner_addends<-1>(a, b, n, blo, alo);
#if ATX_STRICT
  const double h2 = 0.0;
#else
  const double h2 = 0.5 / (1.0 + r.dp);
#endif
  for (int m = 0; m < nslice; m++) {
    for (int j = 0; j < nop; j++) {
      const double len = op[2 + 2 * j];
      if (op[1 + 2 * j] == 0.0) {
        if (RAD) rad_drift(r, len, 1.0 / (1.0 + r.dp)); else fastdrift(r, len * pn0, h2);
      } else {
        if (RAD) {
          double pn = 1.0 / (1.0 + r.dp);
          if (BEND) rad_bnd_kick<-1>(r, a, b, n, blo, alo, len, irho, len * irho, radc, radc * len, pn);
          else rad_str_kick<-1>(r, a, b, n, blo, alo, len, radc, radc * len, pn);
        } else {
          if (BEND) bnd_kick<-1>(r, a, b, n, blo, alo, len, irho, len * irho); else str_kick<-1>(r, a, b, n, blo, alo, len);
        }
      }
    }
  }
  return r;
}

// Particles per lane: the element code below takes the P particles a lane
// tracks as an array and runs every step of a magnet for all of them before
// the next step, so the P independent dependency chains interleave in one
// instruction stream, and the magnet's scalar constants, loop control and
// branches serve P particles. Per-particle maps that are rare or large stay
// out of line and run once per particle.
// The field of a magnet, by the coefficients that are not zero (chosen when the
// lattice is compiled, atx_host.cpp fill_op). Quadrupoles, sextupoles and
// octupoles have one coefficient and a bend often none, so the fast build
// spells their kicks out instead of running Horner over zeros: 2 FP64
// instructions instead of 6 per quadrupole kick, 5 instead of 10 per sextupole
// kick, 8 instead of 14 per octupole kick, 19 instead of 23 per radiating
// quadrupole kick, 20 instead of 33 per kick of a radiating bend without
// gradient. (The VALU issued on 83 % of the cycles of a full device before that,
// so time follows the instruction count.) The strict build evaluates all coefficients.
// A particle whose result is not finite is recomputed with the general form
// (run_turn): zeros times an infinity are NaN there, as in the reference.
enum Form : int {
  F_GENERAL = 0,  // Horner over all coefficients
  F_LEAD = 1,     // B[N] only
  F_LEAD0 = 2,    // B[N], B[0] and A[0] (a sextupole that is a corrector, too)
  F_NOFIELD = 3   // none: a bend's own curvature
};

#if !ATX_STRICT
// In-magnet drift of the fast build: nlh = nl / (2 (1+delta)) hoisted with
// nl (delta is constant in a non-radiating magnet).
__device__ __forceinline__ void fastdrift_h(R6& r, double nl, double nlh) {
  r.x = __builtin_fma(nl, r.px, r.x);
  r.y = __builtin_fma(nl, r.py, r.y);
  const double p2 = __builtin_fma(r.px, r.px, r.py * r.py);
  r.ct = __builtin_fma(nlh, p2, r.ct);
}

// What a kick of length kl multiplies by, once per magnet. The rounding of
// such a product is the same at every kick of every turn, so it would add up
// over the turns instead of averaging out: its remainder is kept, too, and is
// added where that costs nothing (radiating kicks) or once per magnet
// (kick_rest). Constants that are only added (a dipole in a sextupole) are the
// addends of the field, which kl then multiplies at each kick.
struct Kick {
  double kl, kli;         // length, length times curvature
  double bn;              // B[N]
  double kb, kb2;         // kl B[N], twice that (LEAD0: 2 B[N])
  double b0, a0;          // B[0], A[0]
  double lo;              // remainder of kb (NOFIELD: of kli)
  double rk;              // radiating: RAD_CONST gamma^3 kl (times the field's constant squared)
};

template <bool BEND, int N, int F>
__device__ __forceinline__ Kick kick_of(cdouble* a, cdouble* b, double lead, double kl, double irho,
                                        double radk) {
  Kick k;
  k.kl = kl;
  k.kli = BEND ? kl * irho : 0.0;
  k.kb = k.kb2 = k.b0 = k.a0 = k.lo = 0.0;
  if (F == F_LEAD) {
    k.kb = kl * lead;
    k.kb2 = 2.0 * k.kb;
    k.lo = __builtin_fma(kl, lead, -k.kb);
  }
  if (F == F_NOFIELD) k.lo = __builtin_fma(kl, irho, -k.kli);
  if (F == F_LEAD0) {
    k.kb2 = 2.0 * lead;
    k.b0 = b[0];
    k.a0 = a[0];
    asm("" : "=v"(k.b0) : "0"(k.b0));  // an FMA reads one scalar: horner_addends
    asm("" : "=v"(k.a0) : "0"(k.a0));
  }
  k.rk = radk;
  k.bn = lead;
  if (F == F_LEAD && !BEND) k.rk = radk * (lead * lead);
  if (F == F_NOFIELD) k.rk = radk * (irho * irho);
  return k;
}

// A non-radiating bend with a gradient: kl (re - (delta - x h) h) is
// kl (c x - d) with c = B[1] + h^2 for the magnet and d = h delta for the
// particle, and their remainders.
struct BendGrad {
  double c, c_lo;
  double d, d_lo;
};

__device__ __forceinline__ BendGrad bend_grad(double lead, double irho, double dp) {
  BendGrad g;
  g.c = __builtin_fma(irho, irho, lead);
  g.c_lo = __builtin_fma(irho, irho, lead - g.c);
  g.d = irho * dp;
  g.d_lo = __builtin_fma(irho, dp, -g.d);
  return g;
}

// The remainders of a whole magnet's kicks in one: lo = the sum of theirs, kl =
// of their lengths. Taken at the first kick: a particle that overflows in a strong
// multipole leaves it with coordinates whose powers are far above its kicks.
template <bool BEND, int N, int F>
__device__ __forceinline__ void kick_rest(R6& r, double lo, double kl, double irho,
                                          const BendGrad& g) {
  if (BEND) {
    r.px = __builtin_fma(-kl, __builtin_fma(g.c_lo, r.x, -g.d_lo), r.px);
    if (F == F_LEAD) r.py = __builtin_fma(lo, r.y, r.py);
  } else if (N == 1) {
    r.px = __builtin_fma(-lo, r.x, r.px);
    r.py = __builtin_fma(lo, r.y, r.py);
  } else if (N == 2) {
    r.px = __builtin_fma(-lo, __builtin_fma(r.x, r.x, -(r.y * r.y)), r.px);
    r.py = __builtin_fma(2.0 * lo, r.x * r.y, r.py);
  } else {
    const double x2 = r.x * r.x, y2 = r.y * r.y;
    r.px = __builtin_fma(-lo, r.x * __builtin_fma(-3.0, y2, x2), r.px);
    r.py = __builtin_fma(lo, r.y * __builtin_fma(3.0, x2, -y2), r.py);
  }
}

// driftkick.c:51-115 by form.
template <bool BEND, int N, int F>
__device__ __forceinline__ void kick(R6& r, const Kick& k, cdouble* a, cdouble* b, int n, double blo,
                                     double alo, double irho, const BendGrad& g) {
  if (F == F_GENERAL) {
    if (BEND) bnd_kick<N>(r, a, b, n, blo, alo, k.kl, irho, k.kli);
    else str_kick<N>(r, a, b, n, blo, alo, k.kl);
    return;
  }
  if (BEND) {
    r.px = __builtin_fma(-k.kl, __builtin_fma(g.c, r.x, -g.d), r.px);
    if (F == F_LEAD) r.py = __builtin_fma(k.kb, r.y, r.py);
    r.ct = __builtin_fma(k.kli, r.x, r.ct);
    return;
  }
  double px = r.px, py = r.py;
  if (F == F_LEAD0) {
    // the dipole with the rest of the field: kl B[0] added by itself would round
    // alike at every kick (30 kicks: twice to four times the error)
    static_assert(F != F_LEAD0 || N == 2, "a sextupole");
    const double re = __builtin_fma(k.bn, __builtin_fma(r.x, r.x, -(r.y * r.y)), k.b0);
    const double im = __builtin_fma(k.kb2, r.x * r.y, k.a0);
    px = __builtin_fma(-k.kl, re, px);
    py = __builtin_fma(k.kl, im, py);
  } else if (N == 1) {
    px = __builtin_fma(-k.kb, r.x, px);
    py = __builtin_fma(k.kb, r.y, py);
  } else if (N == 2) {  // z^2 = (x^2 - y^2) + i 2 x y
    px = __builtin_fma(-k.kb, __builtin_fma(r.x, r.x, -(r.y * r.y)), px);
    py = __builtin_fma(k.kb2, r.x * r.y, py);
  } else {  // z^3 = x (x^2 - 3 y^2) + i y (3 x^2 - y^2)
    const double x2 = r.x * r.x, y2 = r.y * r.y;
    px = __builtin_fma(-k.kb, r.x * __builtin_fma(-3.0, y2, x2), px);
    py = __builtin_fma(k.kb, r.y * __builtin_fma(3.0, x2, -y2), py);
  }
  r.px = px;
  r.py = py;
}

// Radiating magnets of the fast build carry the transverse momenta as
// angles x' = px/(1+delta), y' = py/(1+delta) from entry to exit: a drift is
// then x += L x', ct += (L/2)(x'^2 + y'^2), its x'^2 + y'^2 is the kick's
// s2 (the kick that follows a drift sees the same angles), and a kick turns
// px = x'(1+delta') - kl Re, the reference's update, into
// x' <- x' - kl Re / (1+delta'). pn = 1/(1+delta).
struct Ang {
  double xp, yp, s2, pn;
};

__device__ __forceinline__ Ang to_angles(const R6& r) {
  const double pn = fast_rcp(1.0 + r.dp);
  return Ang{r.px * pn, r.py * pn, 0.0, pn};
}

__device__ __forceinline__ void from_angles(R6& r, const Ang& g) {
  const double opd = 1.0 + r.dp;
  r.px = g.xp * opd;
  r.py = g.yp * opd;
}

__device__ __forceinline__ void rad_drift_ang(R6& r, Ang& g, double len, double hlen) {
  r.x = __builtin_fma(len, g.xp, r.x);
  r.y = __builtin_fma(len, g.yp, r.y);
  g.s2 = __builtin_fma(g.xp, g.xp, g.yp * g.yp);
  r.ct = __builtin_fma(hlen, g.s2, r.ct);
}

// diff_str_kick.c:19-83 and diff_bnd_kick.c:85-174 (bdiff == NULL) in angle
// form. w is the radiated fraction, radk b2p factor (1+delta): delta falls by
// w (1+delta), and 1/(1+delta) becomes pn/(1-w) = pn (1 + w + w^2) to a
// relative w^3, below 1e-17 for |w| <= 2e-6. The last kick of a slice (REFRESH)
// takes 1 - (1+delta') pn in the place of w: that holds the rounding errors of
// pn as well, which would otherwise add up over the magnet.
// Straight magnets: the factor (1+s2/2)/(1+s2) is 1 - (s2/2)(1 - s2 + s2^2),
// relative error s2^4/2, below 1e-16 for s2 <= 1e-4 (angles up to 10 mrad).
// CHECKED: lanes outside either range divide instead, under a vote per kick.
// Otherwise the largest s2 and |w| of the magnet are kept, and a magnet in which
// one was outside is run again with the checks (run_turn): no branch and no
// compare in the slices. All other lanes get the same bits either way. The
// largest are kept by their high words, two of them with one v_max3_i32; of
// the kicks of length K1 and K2, whose w have opposite signs, each for itself
// (of negative numbers, too, the high word grows with the magnitude).
struct Largest {
  int s2, w[2];
};
__device__ __forceinline__ int high_word(double v) {
  return (int)(uint32_t)(__builtin_bit_cast(uint64_t, v) >> 32);
}
__device__ __forceinline__ uint64_t outside(const Largest& m) {
  constexpr int kS2 = 0x3F1A36E2, kW = 0x3EC0C6F7;  // of 1e-4 and 2e-6
  return __builtin_amdgcn_ballot_w64(m.s2 >= kS2) |
         __builtin_amdgcn_ballot_w64((m.w[0] & 0x7fffffff) >= kW) |
         __builtin_amdgcn_ballot_w64((m.w[1] & 0x7fffffff) >= kW);
}
template <bool BEND, int N, int F, bool CHECKED, bool REFRESH>
__device__ __forceinline__ void rad_kick_ang(R6& r, Ang& g, const Kick& k, cdouble* a, cdouble* b,
                                             int n, double blo, double alo, double irho,
                                             int& most_s2, int& most_w) {
  const double x = r.x, y = r.y;
  const double s2 = g.s2;
  const double d0 = r.dp;
  const double opd = 1.0 + d0;
  const double ro = k.rk * opd;
  double re = 0.0, im = 0.0;
  if (F == F_GENERAL) field<N>(r, a, b, n, blo, alo, re, im);
  if (BEND && F == F_LEAD) {
    re = k.bn * x;
    im = k.bn * y;
  }
  double w;
  bool odd = false;
  if (BEND) {
    const double hx = __builtin_fma(x, irho, 1.0);
    double b2;  // squared field across the velocity, times its length squared
    if (F == F_NOFIELD) {
      b2 = __builtin_fma(g.xp, g.xp, hx * hx);
    } else {
      const double by = re + irho;
      const double byh = by * hx;
      const double bxh = im * hx;
      const double cr = __builtin_fma(im, g.yp, -by * g.xp);
      b2 = __builtin_fma(cr, cr, __builtin_fma(byh, byh, bxh * bxh));
    }
    const double f = __builtin_fma(0.5, s2, hx) * rcp1(__builtin_fma(hx, hx, s2));
    w = (b2 * ro) * f;  // the reciprocal in f comes last
  } else {
    double b2;
    if (F == F_LEAD) {  // |B|^2 over B[1]^2
      const double cr = __builtin_fma(y, g.yp, -x * g.xp);
      b2 = __builtin_fma(cr, cr, __builtin_fma(x, x, y * y));
    } else {
      const double cr = __builtin_fma(im, g.yp, -re * g.xp);
      b2 = __builtin_fma(cr, cr, __builtin_fma(re, re, im * im));
    }
    const double f = __builtin_fma(s2, __builtin_fma(s2, __builtin_fma(-0.5, s2, 0.5), -0.5), 1.0);
    w = b2 * (f * ro);  // f does not wait for x
    if (CHECKED)
      odd = s2 > 1e-4;
    else
      most_s2 = max(most_s2, high_word(s2));
    if (CHECKED && __builtin_amdgcn_ballot_w64(odd) != 0) {
      const double fw = __builtin_fma(0.5, s2, 1.0) * rcp1(1.0 + s2);
      w = odd ? b2 * (fw * ro) : w;
    }
  }
  r.dp = __builtin_fma(-w, opd, d0);
  const double e = REFRESH ? __builtin_fma(-(1.0 + r.dp), g.pn, 1.0) : w;
  double pn = __builtin_fma(g.pn, __builtin_fma(e, e, e), g.pn);
  if (CHECKED) {
    const bool far = __builtin_fabs(w) > 2e-6;
    if (__builtin_amdgcn_ballot_w64(far) != 0) pn = far ? fast_rcp(1.0 + r.dp) : pn;
  } else {
    most_w = max(most_w, high_word(w));
  }
  if (!BEND && F == F_LEAD) {
    const double kn = __builtin_fma(k.kb, pn, k.lo);  // lo pn, to a relative delta
    g.xp = __builtin_fma(-x, kn, g.xp);
    g.yp = __builtin_fma(y, kn, g.yp);
  } else if (BEND && F == F_NOFIELD) {
    const double u = __builtin_fma(-x, irho, d0);
    g.xp = __builtin_fma(u, __builtin_fma(k.kli, pn, k.lo), g.xp);
    r.ct = __builtin_fma(k.kli, x, r.ct);
  } else {
    const double kn = k.kl * pn;
    double v = re;
    if (BEND) {
      const double u = __builtin_fma(-x, irho, d0);
      v = __builtin_fma(-u, irho, re);
      r.ct = __builtin_fma(k.kli, x, r.ct);
    }
    g.xp = __builtin_fma(-v, kn, g.xp);
    g.yp = __builtin_fma(im, kn, g.yp);
  }
  g.pn = pn;
}
#endif

// Entry and exit of a thick multipole, per particle: FieldScaling, T1/R1,
// apertures, bend edge, quadrupole fringe (StrMPoleSymplectic4Pass.c:57-78,
// 96-104; BndMPoleSymplectic4Pass.c:75-96, 114-122).
// One test for the transforms and apertures an unmisaligned magnet without
// apertures has none of, before the tests of each.
constexpr uint32_t F_ENTRY_ANY = F_T1 | F_R1 | F_RAP | F_EAP;
constexpr uint32_t F_EXIT_ANY = F_R2 | F_T2 | F_RAP | F_EAP | F_SCALE;

// LEAN: without the maps that are functions of their own (F_LEAN).
template <bool BEND, bool LEAN>
__device__ __forceinline__ void mpole_entry(R6& r, cDevElem& h, cdouble* pool, cdouble* s) {
  if (h.flags & F_ENTRY_ANY) {
    if (LEAN) {
      if (h.flags & F_T1) add_t(r, pool + h.t1);
      if (h.flags & F_R1) r = mul_r_inl(r, pool + h.r1);
    } else {
      entry_xform(r, h, pool);
    }
    apertures(r, h, pool);
  }
  if (BEND) edge<LEAN>(r, h.edge & 0xff, s[S_IRHO], s[S_FX_IN], s[S_FY_IN], s[S_EDGE_IN], s[S_CORR_IN], 1.0);
  if (!LEAN && (h.fringe & 0xff)) quad_fringe_in(r, h, pool, s[S_B2]);
}

template <bool BEND, bool LEAN>
__device__ __forceinline__ void mpole_exit(R6& r, cDevElem& h, cdouble* pool, cdouble* s) {
  if (!LEAN && (h.fringe & 0xff00)) quad_fringe_out(r, h, pool, s[S_B2]);
  if (BEND) edge<LEAN>(r, (h.edge >> 8) & 0xff, s[S_IRHO], s[S_FX_OUT], s[S_FY_OUT], s[S_EDGE_OUT], s[S_CORR_OUT], -1.0);
  if (h.flags & F_EXIT_ANY) {
    apertures(r, h, pool);
    if (LEAN) {
      if (h.flags & F_R2) r = mul_r_inl(r, pool + h.r2);
      if (h.flags & F_T2) add_t(r, pool + h.t2);
    } else {
      exit_xform(r, h, pool);
      if (h.flags & F_SCALE) change_pref(r, s[S_INVSCALE]);
    }
  }
}

// Called once all constants of an element have been asked for (its arguments,
// held here so that they have arrived): the loop over the records then asks for
// the next record (run_turn).
struct NotAhead {
  template <class... T>
  __device__ __forceinline__ void operator()(T...) const {}
};
__device__ __forceinline__ void hold(double v) { asm volatile("" ::"s"(v)); }

// Slices of StrMPoleSymplectic4Pass.c:79-93 and BndMPoleSymplectic4Pass.c:97-111
// for the P particles of a lane; U slices per loop iteration. pn = 1/(1+delta)
// at the entry, nl1, nl2 = the drift lengths times it.
// The fast build joins the last drift of a slice and the first of the next
// (delta and the momenta are the same in both): three drifts per slice
// instead of four. The path length is still added drift by drift: the terms of
// a magnet's slices are nearly equal and round alike against a ct a million
// times larger, so known answers of the reference hold that rounding.
template <bool BEND, int N, int F, int P, int U, class Ahead>
__device__ __forceinline__ void mpole_slices(R6* r, cdouble* a, cdouble* b, int n, int nslice,
                                             double lead, const double* nl1, const double* nl2,
                                             double k1, double k2, double irho,
                                             const Ahead& ahead) {
  double blo, alo;
  horner_addends<N>(a, b, n, blo, alo);
  if (F == F_GENERAL && N == 3) ahead(k1, k2, a[3], b[3], a[2], b[2], a[1], b[1], a[0], b[0]);
  else if (F == F_GENERAL && N == 2) ahead(k1, k2, a[2], b[2], a[1], b[1], a[0], b[0]);
  else if (F == F_GENERAL && N == 1) ahead(k1, k2, a[1], b[1], a[0], b[0]);
  else if (F == F_LEAD0) ahead(k1, k2, a[0], b[0]);
  else ahead(k1, k2);
#if ATX_STRICT
  const double ki1 = k1 * irho, ki2 = k2 * irho;
  // U slices per iteration: a constant-count inner loop, fully unrolled
  // (the slices may hold wave-wide votes, which a runtime-count unroll
  // cannot duplicate), then the remaining slices one by one
  auto slice = [&]() {
#pragma unroll
    for (int q = 0; q < P; q++) fastdrift(r[q], nl1[q], 0.0);
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (BEND) bnd_kick<N>(r[q], a, b, n, blo, alo, k1, irho, ki1); else str_kick<N>(r[q], a, b, n, blo, alo, k1);
    }
#pragma unroll
    for (int q = 0; q < P; q++) fastdrift(r[q], nl2[q], 0.0);
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (BEND) bnd_kick<N>(r[q], a, b, n, blo, alo, k2, irho, ki2); else str_kick<N>(r[q], a, b, n, blo, alo, k2);
    }
#pragma unroll
    for (int q = 0; q < P; q++) fastdrift(r[q], nl2[q], 0.0);
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (BEND) bnd_kick<N>(r[q], a, b, n, blo, alo, k1, irho, ki1); else str_kick<N>(r[q], a, b, n, blo, alo, k1);
    }
#pragma unroll
    for (int q = 0; q < P; q++) fastdrift(r[q], nl1[q], 0.0);
  };
  int m = 0;
  for (; m + U <= nslice; m += U) {
#pragma unroll
    for (int u = 0; u < U; u++) slice();
  }
  for (; m < nslice; m++) slice();
#else
  const Kick c1 = kick_of<BEND, N, F>(a, b, lead, k1, irho, 0.0);
  const Kick c2 = kick_of<BEND, N, F>(a, b, lead, k2, irho, 0.0);
  double nh1[P], nh2[P], nl12[P];  // delta is constant through the slices
  BendGrad bg[P] = {};
#pragma unroll
  for (int q = 0; q < P; q++) {
    if (BEND && F != F_GENERAL) bg[q] = bend_grad(F == F_LEAD ? lead : 0.0, irho, r[q].dp);
    const double h2 = 0.5 * fast_rcp(1.0 + r[q].dp);
    nh1[q] = nl1[q] * h2;
    nh2[q] = nl2[q] * h2;
    nl12[q] = 2.0 * nl1[q];
  }
  auto drift = [&](const double* nl, const double* nh) {
#pragma unroll
    for (int q = 0; q < P; q++) fastdrift_h(r[q], nl[q], nh[q]);
  };
  auto drift2 = [&]() {  // the last drift of a slice and the first of the next
#pragma unroll
    for (int q = 0; q < P; q++) {
      fastdrift_h(r[q], nl12[q], nh1[q]);
      r[q].ct = __builtin_fma(nh1[q], __builtin_fma(r[q].px, r[q].px, r[q].py * r[q].py), r[q].ct);
    }
  };
  auto kicks = [&](const Kick& c) {
#pragma unroll
    for (int q = 0; q < P; q++) kick<BEND, N, F>(r[q], c, a, b, n, blo, alo, irho, bg[q]);
  };
  auto body = [&]() {  // a slice without its outer drifts
    kicks(c1);
    drift(nl2, nh2);
    kicks(c2);
    drift(nl2, nh2);
    kicks(c1);
  };
  drift(nl1, nh1);
  if (F == F_LEAD || F == F_NOFIELD) {
    const double lo = (2.0 * c1.lo + c2.lo) * (double)nslice;
    const double kl = (2.0 * k1 + k2) * (double)nslice;
#pragma unroll
    for (int q = 0; q < P; q++) kick_rest<BEND, N, F>(r[q], lo, kl, irho, bg[q]);
  }
  int m = 1;
  for (; m + U <= nslice; m += U) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      body();
      drift2();
    }
  }
  for (; m < nslice; m++) {
    body();
    drift2();
  }
  body();
  drift(nl1, nh1);
#endif
}

// Slices of StrMPoleSymplectic4RadPass.c:83-99 and
// BndMPoleSymplectic4RadPass.c:98-112, likewise. CHECKED, bad: rad_kick_ang.
template <bool BEND, int N, int F, int P, int U, bool CHECKED, class Ahead>
__device__ __forceinline__ void mpole_rad_slices(R6* r, cdouble* a, cdouble* b, int n, int nslice,
                                                 double lead, double l1, double l2, double k1,
                                                 double k2, double irho, double radc, double rk1, double rk2,
                                                 uint64_t& bad, const Ahead& ahead) {
  double blo, alo;
  horner_addends<N>(a, b, n, blo, alo);
  const double rk = ATX_STRICT ? radc : rk1;
  if (F == F_GENERAL && N == 3)
    ahead(l1, l2, k1, k2, rk, rk2, a[3], b[3], a[2], b[2], a[1], b[1], a[0], b[0]);
  else if (F == F_GENERAL && N == 2)
    ahead(l1, l2, k1, k2, rk, rk2, a[2], b[2], a[1], b[1], a[0], b[0]);
  else if (F == F_GENERAL && N == 1) ahead(l1, l2, k1, k2, rk, rk2, a[1], b[1], a[0], b[0]);
  else ahead(l1, l2, k1, k2, rk, rk2);
#if ATX_STRICT
  const double ki1 = k1 * irho, ki2 = k2 * irho;
  // 1/(1+delta), divided as the reference does; delta changes in the kicks only,
  // so the quotient of one kick is that of the drifts and the kick after it
  double pn[P];
#pragma unroll
  for (int q = 0; q < P; q++) pn[q] = 1.0 / (1.0 + r[q].dp);
  // U slices per iteration: a constant-count inner loop, fully unrolled
  // (the slices may hold wave-wide votes, which a runtime-count unroll
  // cannot duplicate), then the remaining slices one by one
  auto slice = [&]() {
#pragma unroll
    for (int q = 0; q < P; q++) rad_drift(r[q], l1, pn[q]);
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (BEND) rad_bnd_kick<N>(r[q], a, b, n, blo, alo, k1, irho, ki1, radc, 0.0, pn[q]);
      else rad_str_kick<N>(r[q], a, b, n, blo, alo, k1, radc, 0.0, pn[q]);
    }
#pragma unroll
    for (int q = 0; q < P; q++) rad_drift(r[q], l2, pn[q]);
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (BEND) rad_bnd_kick<N>(r[q], a, b, n, blo, alo, k2, irho, ki2, radc, 0.0, pn[q]);
      else rad_str_kick<N>(r[q], a, b, n, blo, alo, k2, radc, 0.0, pn[q]);
    }
#pragma unroll
    for (int q = 0; q < P; q++) rad_drift(r[q], l2, pn[q]);
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (BEND) rad_bnd_kick<N>(r[q], a, b, n, blo, alo, k1, irho, ki1, radc, 0.0, pn[q]);
      else rad_str_kick<N>(r[q], a, b, n, blo, alo, k1, radc, 0.0, pn[q]);
    }
#pragma unroll
    for (int q = 0; q < P; q++) rad_drift(r[q], l1, pn[q]);
  };
  int m = 0;
  for (; m + U <= nslice; m += U) {
#pragma unroll
    for (int u = 0; u < U; u++) slice();
  }
  for (; m < nslice; m++) slice();
#else
  const Kick c1 = kick_of<BEND, N, F>(a, b, lead, k1, irho, rk1);
  const Kick c2 = kick_of<BEND, N, F>(a, b, lead, k2, irho, rk2);
  const double hl1 = 0.5 * l1, hl2 = 0.5 * l2, l12 = 2.0 * l1;
  Ang g[P];
#pragma unroll
  for (int q = 0; q < P; q++) g[q] = to_angles(r[q]);  // one reciprocal per magnet
  auto drift = [&](double len, double hlen) {
#pragma unroll
    for (int q = 0; q < P; q++) rad_drift_ang(r[q], g[q], len, hlen);
  };
  auto drift2 = [&]() {  // the last drift of a slice and the first of the next
#pragma unroll
    for (int q = 0; q < P; q++) {
      rad_drift_ang(r[q], g[q], l12, hl1);
      r[q].ct = __builtin_fma(hl1, g[q].s2, r[q].ct);
    }
  };
  Largest m = {0, {INT_MIN, INT_MIN}};
  auto kicks = [&](const Kick& c, int& most_w) {
#pragma unroll
    for (int q = 0; q < P; q++)
      rad_kick_ang<BEND, N, F, CHECKED, false>(r[q], g[q], c, a, b, n, blo, alo, irho, m.s2, most_w);
  };
  auto body = [&]() {  // a slice without its outer drifts
    kicks(c1, m.w[0]);
    drift(l2, hl2);
    kicks(c2, m.w[1]);
    drift(l2, hl2);
#pragma unroll
    for (int q = 0; q < P; q++)
      rad_kick_ang<BEND, N, F, CHECKED, true>(r[q], g[q], c1, a, b, n, blo, alo, irho, m.s2, m.w[0]);
  };
  drift(l1, hl1);
  int k = 1;
  for (; k + U <= nslice; k += U) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      body();
      drift2();
    }
  }
  for (; k < nslice; k++) {
    body();
    drift2();
  }
  body();
  drift(l1, hl1);
#pragma unroll
  for (int q = 0; q < P; q++) from_angles(r[q], g[q]);
  if (!CHECKED) bad |= outside(m);
#endif
}

// StrMPoleSymplectic4Pass.c:57-104 and BndMPoleSymplectic4Pass.c:75-122 for
// the P particles of a lane; U slices per loop iteration.
template <bool BEND, int N, int P, int U, bool LEAN>
__device__ __forceinline__ void mpole(R6* r, cDevElem& h, cdouble* pool) {
  cdouble* s = pool + h.sc;
  cdouble* a = pool + h.poly;
  cdouble* b = a + h.order + 1;
  const int n = h.order;
  double pn[P], nl1[P], nl2[P];
#pragma unroll
  for (int q = 0; q < P; q++) {
    if (!LEAN && (h.flags & F_SCALE)) change_pref(r[q], s[S_SCALE]);
#if ATX_STRICT
    pn[q] = 1.0 / (1.0 + r[q].dp);  // before T1/R1, as the reference hoists it
#else
    pn[q] = fast_rcp(1.0 + r[q].dp);  // before T1/R1, as the reference hoists it
#endif
    nl1[q] = s[S_L1] * pn[q];
    nl2[q] = s[S_L2] * pn[q];
    mpole_entry<BEND, LEAN>(r[q], h, pool, s);
  }
  const double irho = s[S_IRHO];
  if (!LEAN && h.ops >= 0) {
#pragma unroll
    for (int q = 0; q < P; q++)
      r[q] = slices_ops<BEND, false>(r[q], a, b, n, pool + h.ops, h.nslice, pn[q], irho, 0.0);
  } else if (h.nslice > 0) {
    mpole_slices<BEND, N, F_GENERAL, P, U>(r, a, b, n, h.nslice, 0.0, nl1, nl2, s[S_K1], s[S_K2], irho,
                                          NotAhead());
  }
#pragma unroll
  for (int q = 0; q < P; q++) mpole_exit<BEND, LEAN>(r[q], h, pool, s);
}

// StrMPoleSymplectic4RadPass.c:61-110 and BndMPoleSymplectic4RadPass.c:76-123
// for the P particles of a lane; U slices per loop iteration.
template <bool BEND, int N, int P, int U, bool LEAN>
__device__ __forceinline__ void mpole_rad(R6* r, cDevElem& h, cdouble* pool) {
  cdouble* s = pool + h.sc;
  cdouble* a = pool + h.poly;
  cdouble* b = a + h.order + 1;
  const int n = h.order;
#pragma unroll
  for (int q = 0; q < P; q++) {
    if (!LEAN && (h.flags & F_SCALE)) change_pref(r[q], s[S_SCALE]);
    mpole_entry<BEND, LEAN>(r[q], h, pool, s);
  }
  const double irho = s[S_IRHO];
  const double radc = s[S_RADC];
  if (!LEAN && h.ops >= 0) {
#pragma unroll
    for (int q = 0; q < P; q++)
      r[q] = slices_ops<BEND, true>(r[q], a, b, n, pool + h.ops, h.nslice, 0.0, irho, radc);
  } else if (h.nslice > 0) {
    uint64_t bad = 0;
    mpole_rad_slices<BEND, N, F_GENERAL, P, U, true>(r, a, b, n, h.nslice, 0.0, s[S_L1], s[S_L2], s[S_K1],
                                                     s[S_K2], irho, radc, s[S_RK1], s[S_RK2], bad,
                                                     NotAhead());
  }
#pragma unroll
  for (int q = 0; q < P; q++) mpole_exit<BEND, LEAN>(r[q], h, pool, s);
}

// Pointers that every lane of the wave holds alike, back in scalar registers
// (arguments of a function that is not inlined arrive in vector registers).
template <typename T>
__device__ __forceinline__ T uniform(T p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (T)(((uint64_t)hi << 32) | lo);
}

// Elements by their headers run out of line, one function per kind and order:
// the loop over the records then keeps its registers (and its code, which
// has to stay in the instruction cache) for the common ops. A call costs about
// 0.4 us with one wave per SIMD (the callee saves the scalar registers it
// uses), so what has a record runs inline: multipoles of orders above 3 and of
// other integrators, misaligned elements of other kinds, cavities and the exact
// passes are left.
template <bool BEND, bool RAD, int N, int U, bool LEAN>
__device__ __noinline__ R6 mpole_call(R6 r, cDevElem* hp, cdouble* poolp) {
  cDevElem& h = *uniform(hp);
  cdouble* pool = uniform(poolp);
  if (RAD) mpole_rad<BEND, N, 1, U, LEAN>(&r, h, pool); else mpole<BEND, N, 1, U, LEAN>(&r, h, pool);
  return r;
}

template <bool BEND, bool RAD, int U, bool LEAN>
__device__ __forceinline__ R6 mpole_order(const R6& r, cDevElem& h, cdouble* pool) {
  switch (h.order) {
    case 0: return mpole_call<BEND, RAD, 0, U, LEAN>(r, &h, pool);
    case 1: return mpole_call<BEND, RAD, 1, U, LEAN>(r, &h, pool);
    case 2: return mpole_call<BEND, RAD, 2, U, LEAN>(r, &h, pool);
    case 3: return mpole_call<BEND, RAD, 3, U, LEAN>(r, &h, pool);
    default: return mpole_call<BEND, RAD, -1, U, LEAN>(r, &h, pool);
  }
}

// A function that calls others keeps its return address in scratch memory
// over the calls, so the magnets without such maps have functions without.
template <bool BEND, bool RAD, int U>
__device__ __forceinline__ R6 mpole_dispatch(const R6& r, cDevElem& h, cdouble* pool) {
  if (h.flags & F_LEAN) return mpole_order<BEND, RAD, U, true>(r, h, pool);
  return mpole_order<BEND, RAD, U, false>(r, h, pool);
}

// ThinMPolePass.c:42-63
__device__ __forceinline__ void thin(R6& r, cDevElem& h, cdouble* pool) {
  cdouble* s = pool + h.sc;
  cdouble* a = pool + h.poly;
  cdouble* b = a + h.order + 1;
  if (h.flags & F_SCALE) change_pref(r, s[S_SCALE]);
  entry_xform(r, h, pool);
  apertures(r, h, pool);
  switch (h.order) {
    case 0: str_kick<0>(r, a, b, 0, 0.0, 0.0, 1.0); break;
    case 1: str_kick<1>(r, a, b, 1, b[0], a[0], 1.0); break;
    case 2: str_kick<2>(r, a, b, 2, b[1], a[1], 1.0); break;
    case 3: str_kick<3>(r, a, b, 3, b[2], a[2], 1.0); break;
    default: str_kick<-1>(r, a, b, h.order, 0.0, 0.0, 1.0); break;
  }
  const double bax = s[S_BAX], bay = s[S_BAY];
  r.px += bax * r.dp;
  r.py -= bay * r.dp;
  r.ct -= bax * r.x - bay * r.y;
  exit_xform(r, h, pool);
  if (h.flags & F_SCALE) change_pref(r, s[S_INVSCALE]);
}

// attrackfunc.c:5-42: hft = h/f - T0 prepared on the host. The sine is the
// host C library's, restated bit for bit (atx_libm.h), in both builds.
__device__ __noinline__ double rf_kick(double ct, double nv, double twopif, double lag,
                                       double hft0, double philag, double nt) {
#pragma clang fp contract(off)
  return -nv * libm::host_sin(twopif * ((ct - lag) / 2.99792458e8 - hft0 * nt) - philag);
}

__device__ __forceinline__ void rf_cavity(R6& r, cDevElem& h, cdouble* pool, int nturn) {
  cdouble* s = pool + h.sc;
  const double nt = (double)nturn;
  if (!(h.flags & F_THICK)) {
    if (h.flags & F_RFKICK)
      r.dp += rf_kick(r.ct, s[S_RF_NV], s[S_RF_TWOPIF], s[S_RF_LAG], s[S_RF_HFT0], s[S_RF_PHILAG], nt);
  } else {
    drift6(r, s[S_RF_HALF]);
    if (h.flags & F_RFKICK)
      r.dp += rf_kick(r.ct, s[S_RF_NV], s[S_RF_TWOPIF], s[S_RF_LAG], s[S_RF_HFT0], s[S_RF_PHILAG], nt);
    drift6(r, s[S_RF_HALF]);
  }
}

// CavityPass.c:18-56: no turn dependence (nv = V/E prepared on the host).
__device__ __noinline__ R6 cavity(R6 r, cdouble* s, bool thick) {
  if (thick) drift6(r, s[S_RF_HALF]);
  r.dp += -s[S_RF_NV] *
          libm::host_sin(s[S_RF_TWOPIF] * (r.ct - s[S_RF_LAG]) / 2.99792458e8 - s[S_RF_PHILAG]);
  if (thick) drift6(r, s[S_RF_HALF]);
  return r;
}

// Exact drift, absolute path length (exactdrift.c:4-16).
__device__ __forceinline__ void exact_drift(R6& r, double L) {
  const double opd = 1.0 + r.dp;
  const double pz = sqrt(opd * opd - r.px * r.px - r.py * r.py);
  const double nl = L / pz;
  r.x += r.px * nl;
  r.y += r.py * nl;
  r.ct += nl * opd;
}

// The same drift in the form of the radiating pass (diff_exactdrift.c:30-43).
__device__ __forceinline__ void exact_rad_drift(R6& r, double L) {
  const double pn = 1.0 / (1.0 + r.dp);
  const double xpr = r.px * pn;
  const double ypr = r.py * pn;
  const double nl = L * pn / sqrt(1.0 - xpr * xpr - ypr * ypr);
  r.x += nl * r.px;
  r.y += nl * r.py;
  r.ct += nl * (1.0 + r.dp);
}

// Radiating straight kick with the exact velocity (diff_str_exactkick.c:14-71).
__device__ __forceinline__ void exact_rad_kick(R6& r, cdouble* a, cdouble* b, int n, double kl,
                                               double radc) {
  double re, im;
  field<-1>(r, a, b, n, 0.0, 0.0, re, im);
  double pn = 1.0 / (1.0 + r.dp);
  const double xpr = r.px * pn;
  const double ypr = r.py * pn;
  const double t = im * xpr + re * ypr;
  const double b2p = im * im + re * re - t * t;
  const double factor = kl / (pn * pn) / sqrt(1.0 - xpr * xpr - ypr * ypr);
  r.dp -= radc * b2p * factor;
  pn = 1.0 / (1.0 + r.dp);
  r.px = xpr / pn;
  r.py = ypr / pn;
  r.px -= kl * re;
  r.py += kl * im;
}

// PTC multipole fringe (Forest 13.29) of every order, edge = +1 at the
// entrance, -1 at the exit (exactmultipolefringe.c:2-95, skip_b0 = 0).
__device__ __noinline__ R6 multipole_fringe(R6 r, cdouble* pa, cdouble* pb, int order, double edge) {
  double fx = 0, fy = 0, fx_x = 0, fx_y = 0, fy_x = 0, fy_y = 0;
  double rx = 1.0, ix = 0.0;
  for (int k = 0; k <= order; k++) {
    const double bn = pb[k], an = pa[k];
    const int j = k + 1;
    const double drx = rx, dix = ix;
    rx = drx * r.x - dix * r.y;
    ix = drx * r.y + dix * r.x;
    double u = bn * rx - an * ix;
    double v = bn * ix + an * rx;
    double du = bn * drx - an * dix;
    double dv = bn * dix + an * drx;
    const double f1 = -edge / 4.0 / (j + 1);
    u = u * f1;
    v = v * f1;
    du = du * f1;
    dv = dv * f1;
    const double dux = j * du, dvx = j * dv, duy = -j * dv, dvy = j * du;
    const double nf = 1.0 * (j + 2) / j;
    fx += u * r.x + nf * v * r.y;
    fy += u * r.y - nf * v * r.x;
    fx_x += dux * r.x + u + nf * r.y * dvx;
    fx_y += duy * r.x + nf * v + nf * r.y * dvy;
    fy_x += dux * r.y - nf * v - nf * r.x * dvx;
    fy_y += duy * r.y + u - nf * r.x * dvy;
  }
  const double del = 1.0 / (1 + r.dp);
  const double ma = 1 - fx_x * del;
  const double mb = -fy_x * del;
  const double md = 1 - fy_y * del;
  const double mc = -fx_y * del;
  r.x = r.x - fx * del;
  r.y = r.y - fy * del;
  const double pxf = (md * r.px - mb * r.py) / (ma * md - mb * mc);
  const double pyf = (ma * r.py - mc * r.px) / (ma * md - mb * mc);
  r.py = pyf;
  r.px = pxf;
  r.ct = r.ct - (r.px * fx + r.py * fy) * del * del;
  return r;
}

// ExactMultipolePass.c:27-96 / ExactMultipoleRadPass.c:26-104 slices, out
// of line (generic order): these passes are rare in rings.
__device__ __noinline__ R6 exact_slices(R6 r, cdouble* a, cdouble* b, int n, int nslice,
                                        cdouble* s, bool rad) {
  const double l1 = s[S_L1], l2 = s[S_L2], k1 = s[S_K1], k2 = s[S_K2];
  if (rad) {
    const double radc = s[S_RADC];
    for (int m = 0; m < nslice; m++) {
      exact_rad_drift(r, l1);
      exact_rad_kick(r, a, b, n, k1, radc);
      exact_rad_drift(r, l2);
      exact_rad_kick(r, a, b, n, k2, radc);
      exact_rad_drift(r, l2);
      exact_rad_kick(r, a, b, n, k1, radc);
      exact_rad_drift(r, l1);
    }
  } else {
    for (int m = 0; m < nslice; m++) {
      exact_drift(r, l1);
      str_kick<-1>(r, a, b, n, 0.0, 0.0, k1);
      exact_drift(r, l2);
      str_kick<-1>(r, a, b, n, 0.0, 0.0, k2);
      exact_drift(r, l2);
      str_kick<-1>(r, a, b, n, 0.0, 0.0, k1);
      exact_drift(r, l1);
    }
  }
  return r;
}

__device__ __forceinline__ void exact_mpole(R6& r, cDevElem& h, cdouble* pool, bool rad) {
  cdouble* s = pool + h.sc;
  cdouble* a = pool + h.poly;
  cdouble* b = a + h.order + 1;
  if (h.flags & F_SCALE) change_pref(r, s[S_SCALE]);
  entry_xform(r, h, pool);
  apertures(r, h, pool);
  if (h.fringe & 0xff) r = multipole_fringe(r, a, b, h.order, 1.0);
  r = exact_slices(r, a, b, h.order, h.nslice, s, rad);
  r.ct -= s[S_ELEN];  // absolute path length -> path lengthening
  if (h.fringe & 0xff00) r = multipole_fringe(r, a, b, h.order, -1.0);
  apertures(r, h, pool);
  exit_xform(r, h, pool);
  if (h.flags & F_SCALE) change_pref(r, s[S_INVSCALE]);
}

// Thick corrector without misalignment (CorrectorPass.c:55-89); q0 = xk*xk/3
// + yk*yk/3, the sum's first two terms; nl = L pn, pn = 1/(1+delta).
__device__ __forceinline__ void corrector_map(R6& r, double xk, double yk, double q0, double nl,
                                              double pn) {
  r.ct += nl * pn * (q0 + r.px * r.px + r.py * r.py + r.px * xk + r.py * yk) / 2.0;
  r.x += nl * (r.px + xk / 2.0);
  r.px += xk;
  r.y += nl * (r.py + yk / 2.0);
  r.py += yk;
}

__device__ __forceinline__ double rcp_opd(const R6& r) {
#if ATX_STRICT
  return 1.0 / (1.0 + r.dp);
#else
  return fast_rcp(1.0 + r.dp);
#endif
}

// CorrectorPass.c:25-90
__device__ __forceinline__ void corrector(R6& r, cDevElem& h, cdouble* pool) {
  cdouble* s = pool + h.sc;
  const double xk = s[S_C_XK], yk = s[S_C_YK];
  if (h.flags & F_SCALE) change_pref(r, s[S_SCALE]);
  if (!(h.flags & F_THICK)) {
    entry_xform(r, h, pool);
    apertures(r, h, pool);
    r.px += xk;
    r.py += yk;
  } else {
    const double pn = rcp_opd(r);
    const double nl = s[S_C_LEN] * pn;
    entry_xform(r, h, pool);
    apertures(r, h, pool);
    corrector_map(r, xk, yk, s[S_C_Q0], nl, pn);
    apertures(r, h, pool);
  }
  exit_xform(r, h, pool);
  if (h.flags & F_SCALE) change_pref(r, s[S_INVSCALE]);
}

#if ATX_AUX  // diffusion matrices: built with the reference operation order only
// --- Diffusion matrices -----------------------------------------------------
// Restatement of the reference's Ohmi diffusion-matrix propagation
// (diff_drift.c, diff_thinkick.c, diff_str_kick.c, diff_bnd_kick.c,
// diff_bend_fringe.c, diff_exactdrift.c, diff_str_exactkick.c and
// ATsandwichmmt/ATaddmm of atlalib.c:92-158), used with bdiff != NULL by
// the radiating passes. Matrices are column-major, [i][j] at [i + 6 j], and
// the products keep the reference summation order.

// Entries of a 6x6 matrix that a map fills besides the unit diagonal, as bits.
template <class... I>
constexpr uint64_t entries(I... i) {
  return ((1ull << i) | ...);
}

// B <- M B M^T (atlalib.c:129-147), M the identity and the entries `FILLED`. The
// products with its zeros and ones are left out, the others are summed in the
// reference's order: 84 operations for a drift and 72 for a kick instead of 432.
// The kernel is one chain of them per lane, seven per slice (2,241 elements:
// 73 us, 136 with all products). DENSE: with all, for a matrix that is not
// finite, where zero times an infinity counts.
template <uint64_t FILLED, bool DENSE>
__device__ __forceinline__ void sandwich(const double* m, double* b) {
  double t[36];
#pragma unroll
  for (int i = 0; i < 6; i++) {
#pragma unroll
    for (int j = 0; j < 6; j++) {
      double c = 0;
      bool some = DENSE;
#pragma unroll
      for (int k = 0; k < 6; k++) {
        if (!DENSE && j != k && !((FILLED >> (j + 6 * k)) & 1)) continue;
        const double v = (DENSE || j != k) ? m[j + 6 * k] * b[k + 6 * i] : b[k + 6 * i];
        c = some ? c + v : v;
        some = true;
      }
      t[j + 6 * i] = c;
    }
  }
#pragma unroll
  for (int i = 0; i < 6; i++) {
#pragma unroll
    for (int j = 0; j < 6; j++) {
      double c = 0;
      bool some = DENSE;
#pragma unroll
      for (int k = 0; k < 6; k++) {
        if (!DENSE && j != k && !((FILLED >> (j + 6 * k)) & 1)) continue;
        const double v = (DENSE || j != k) ? t[i + 6 * k] * m[j + 6 * k] : t[i + 6 * k];
        c = some ? c + v : v;
        some = true;
      }
      b[i + 6 * j] = c;
    }
  }
}

__device__ __forceinline__ void eye6(double* m) {
#pragma unroll
  for (int i = 0; i < 36; i++) m[i] = 0.0;
#pragma unroll
  for (int i = 0; i < 6; i++) m[7 * i] = 1.0;
}

// diff_drift.c:2-43
template <bool DENSE>
__device__ __forceinline__ void d_drift(R6& r, double L, double* b) {
  const double pn = 1.0 / (1.0 + r.dp);
  const double xpr = r.px * pn;
  const double ypr = r.py * pn;
  const double nl = L * pn;
  double m[36];
  eye6(m);
  m[6] = nl;
  m[20] = nl;
  m[24] = -nl * xpr;
  m[26] = -nl * ypr;
  m[11] = nl * xpr;
  m[23] = nl * ypr;
  m[29] = -nl * (xpr * xpr + ypr * ypr);
  sandwich<entries(6, 20, 24, 26, 11, 23, 29), DENSE>(m, b);
  r.x += nl * r.px;
  r.y += nl * r.py;
  r.ct += nl * pn * (r.px * r.px + r.py * r.py) / 2.0;
}

// diff_exactdrift.c:2-43
template <bool DENSE>
__device__ __forceinline__ void d_exact_drift(R6& r, double L, double* b) {
  const double pn = 1.0 / (1.0 + r.dp);
  const double xpr = r.px * pn;
  const double ypr = r.py * pn;
  const double nl = L * pn / sqrt(1.0 - xpr * xpr - ypr * ypr);
  const double den = 1.0 - xpr * xpr - ypr * ypr;
  double m[36];
  eye6(m);
  m[6] = nl * (1.0 - ypr * ypr) / den;
  m[18] = nl * xpr * ypr / den;
  m[24] = -nl * xpr / den;
  m[8] = nl * xpr * ypr / den;
  m[20] = nl * (1.0 - xpr * xpr) / den;
  m[26] = -nl * ypr / den;
  m[11] = nl * xpr / den;
  m[23] = nl * ypr / den;
  m[29] = -nl * (xpr * xpr + ypr * ypr) / den;
  sandwich<entries(6, 18, 24, 8, 20, 26, 11, 23, 29), DENSE>(m, b);
  r.x += nl * r.px;
  r.y += nl * r.py;
  r.ct += nl * (1.0 + r.dp);
}

// thinkickM of diff_thinkick.c:1-35 (irho = 0) and diff_bnd_kick.c:1-46
template <bool DENSE>
__device__ __forceinline__ void d_kick_m(const R6& r, cdouble* a, cdouble* bp, int n, double L,
                                         double irho, bool bend, double* b) {
  double imn = n * a[n];
  double ren = n * bp[n];
  for (int k = n - 1; k > 0; k--) {
    const double t = (ren * r.x - imn * r.y) + k * bp[k];
    imn = imn * r.x + ren * r.y + k * a[k];
    ren = t;
  }
  double m[36];
  eye6(m);
  m[1] = -L * ren;
  m[13] = L * imn;
  m[3] = L * imn;
  m[15] = L * ren;
  if (bend) {
    m[25] = L * irho;
    m[1] += -L * irho * irho;
    m[5] = L * irho;
  }
  sandwich<entries(1, 13, 3, 15, 25, 5), DENSE>(m, b);
}

// thinkickB (diff_thinkick.c:37-71, diff_bnd_kick.c:48-83)
__device__ __forceinline__ void d_kick_b(const R6& r, double difc, double b2p, double factor,
                                         double* b) {
  const double pn = 1.0 / (1.0 + r.dp);
  const double pn2 = pn * pn;
  const double b3p = b2p * sqrt(b2p);
  const double bb = difc * b3p * factor / pn2;
  double a[36];
#pragma unroll
  for (int i = 0; i < 36; i++) a[i] = 0.0;
  a[7] = bb * (r.px * r.px) * pn2;
  a[19] = bb * r.px * r.py * pn2;
  a[9] = a[19];
  a[21] = bb * (r.py * r.py) * pn2;
  a[10] = bb * r.px * pn;
  a[25] = a[10];
  a[22] = bb * r.py * pn;
  a[27] = a[22];
  a[28] = bb;
#pragma unroll
  for (int i = 0; i < 6; i++)
#pragma unroll
    for (int j = 0; j < 6; j++) b[i + 6 * j] += a[i + 6 * j];
}

// diff_str_kick.c:19-83 (bend = false), diff_bnd_kick.c:101-174 (bend = true)
template <bool DENSE>
__device__ __forceinline__ void d_rad_kick(R6& r, cdouble* a, cdouble* bp, int n, double L,
                                           double irho, double radc, double difc, bool bend,
                                           double* b) {
  double re = bp[n], im = a[n];
  for (int k = n - 1; k >= 0; k--) {
    const double t = re * r.x - im * r.y + bp[k];
    im = im * r.x + re * r.y + a[k];
    re = t;
  }
  double pn = 1.0 / (1.0 + r.dp);
  const double x = r.x;
  const double xpr = r.px * pn;
  const double ypr = r.py * pn;
  double b2p, factor;
  if (bend) {
    const double by = re + irho, bx = im;
    const double hx = 1 + x * irho;
    const double vn2 = 1.0 / ((1.0 + x * irho) * (1.0 + x * irho) + xpr * xpr + ypr * ypr);
    b2p = ((by * hx) * (by * hx) + (bx * hx) * (bx * hx) + (bx * ypr - by * xpr) * (bx * ypr - by * xpr)) * vn2;
    factor = (1.0 + x * irho + (xpr * xpr + ypr * ypr) / 2.0) / (pn * pn) * L;
  } else {
    const double vn2 = 1.0 / (1.0 + xpr * xpr + ypr * ypr);
    const double cr = im * ypr - re * xpr;
    b2p = (re * re + im * im + cr * cr) * vn2;
    factor = (1.0 + (xpr * xpr + ypr * ypr) / 2.0) / (pn * pn) * L;
  }
  d_kick_m<DENSE>(r, a, bp, n, L, irho, bend, b);
  d_kick_b(r, difc, b2p, factor, b);
  const double d0 = r.dp;
  r.dp -= radc * b2p * factor;
  pn = 1.0 / (1.0 + r.dp);
  r.px = xpr / pn;
  r.py = ypr / pn;
  if (bend) {
    r.px -= L * (re - (d0 - r.x * irho) * irho);
    r.py += L * im;
    r.ct += L * irho * r.x;
  } else {
    r.px -= L * re;
    r.py += L * im;
  }
}

// diff_str_exactkick.c:14-71
template <bool DENSE>
__device__ __forceinline__ void d_exact_rad_kick(R6& r, cdouble* a, cdouble* bp, int n, double L,
                                                 double radc, double difc, double* b) {
  double re = bp[n], im = a[n];
  for (int k = n - 1; k >= 0; k--) {
    const double t = re * r.x - im * r.y + bp[k];
    im = im * r.x + re * r.y + a[k];
    re = t;
  }
  double pn = 1.0 / (1.0 + r.dp);
  const double xpr = r.px * pn;
  const double ypr = r.py * pn;
  const double t = im * xpr + re * ypr;
  const double b2p = im * im + re * re - t * t;
  const double factor = L / (pn * pn) / sqrt(1.0 - xpr * xpr - ypr * ypr);
  d_kick_m<DENSE>(r, a, bp, n, L, 0.0, false, b);
  d_kick_b(r, difc, b2p, factor, b);
  r.dp -= radc * b2p * factor;
  pn = 1.0 / (1.0 + r.dp);
  r.px = xpr / pn;
  r.py = ypr / pn;
  r.px -= L * re;
  r.py += L * im;
}

// diff_bend_fringe.c:2-53; mode and constants as for tracking
__device__ __forceinline__ void d_edge(R6& r, int mode, double irho, double fx, double c0,
                                       double edge_angle, double psi, double sgn, bool bterm,
                                       double* b) {
  const double pn = 1.0 / (1.0 + r.dp);
  double fy;
  if (mode == E_CONST)
    fy = c0;
  else if (mode == E_DIVP)
    fy = c0 / (1.0 + r.dp);
  else if (mode == E_MULPN)
    fy = c0 * pn;
  else
    fy = edge_fy_tan(mode, r.dp, r.px, irho, edge_angle, psi, sgn);
#pragma unroll
  for (int m = 0; m < 6; m++) {
    b[1 + 6 * m] += fx * b[6 * m];
    b[3 + 6 * m] -= fy * b[2 + 6 * m];
  }
  if (bterm)
#pragma unroll
    for (int m = 0; m < 6; m++)
      b[3 + 6 * m] -= b[4 + 6 * m] * r.y * (irho * irho + fy * fy) * psi * pn * pn / irho;
#pragma unroll
  for (int m = 0; m < 6; m++) {
    b[m + 6 * 1] += fx * b[m + 6 * 0];
    b[m + 6 * 3] -= fy * b[m + 6 * 2];
  }
  if (bterm)
#pragma unroll
    for (int m = 0; m < 6; m++)
      b[m + 6 * 3] -= b[m + 6 * 4] * r.y * (irho * irho + fy * fy) * psi * pn * pn / irho;
  r.px += r.x * fx;
  r.py -= r.y * fy;
}

// One radiating element from its entrance orbit: the path of
// StrMPoleSymplectic4RadPass.c:61-110, BndMPoleSymplectic4RadPass.c:76-123
// and ExactMultipoleRadPass.c:56-94 with the matrix updates.
template <bool DENSE>
__device__ __noinline__ void diffusion_elem(R6 r, cDevElem& h, cdouble* pool, double* b) {
  cdouble* s = pool + h.sc;
  cdouble* a = pool + h.poly;
  cdouble* bp = a + h.order + 1;
  const int n = h.order;
  const bool bend = h.kind == K_BNDRAD;
  const bool exact = h.kind == K_EXMPOLERAD;
  const double irho = s[S_IRHO];
  const double radc = s[S_RADC], difc = s[S_DIFC];
  const double l1 = s[S_L1], l2 = s[S_L2], k1 = s[S_K1], k2 = s[S_K2];
  if (h.flags & F_SCALE) change_pref(r, s[S_SCALE]);
  entry_xform(r, h, pool);
  apertures(r, h, pool);
  if (exact) {
    if (h.fringe & 0xff) r = multipole_fringe(r, a, bp, n, 1.0);
    for (int m = 0; m < h.nslice; m++) {
      d_exact_drift<DENSE>(r, l1, b);
      d_exact_rad_kick<DENSE>(r, a, bp, n, k1, radc, difc, b);
      d_exact_drift<DENSE>(r, l2, b);
      d_exact_rad_kick<DENSE>(r, a, bp, n, k2, radc, difc, b);
      d_exact_drift<DENSE>(r, l2, b);
      d_exact_rad_kick<DENSE>(r, a, bp, n, k1, radc, difc, b);
      d_exact_drift<DENSE>(r, l1, b);
    }
    return;  // the exit maps do not change B
  }
  if (bend)
    d_edge(r, h.edge & 0xff, irho, s[S_FX_IN], s[S_FY_IN], s[S_EDGE_IN], s[S_CORR_IN], 1.0,
           (h.flags & F_EDGEB_IN) != 0, b);
  if (h.fringe & 0xff) quad_fringe_in(r, h, pool, s[S_B2]);
  for (int m = 0; m < h.nslice; m++) {
    d_drift<DENSE>(r, l1, b);
    d_rad_kick<DENSE>(r, a, bp, n, k1, irho, radc, difc, bend, b);
    d_drift<DENSE>(r, l2, b);
    d_rad_kick<DENSE>(r, a, bp, n, k2, irho, radc, difc, bend, b);
    d_drift<DENSE>(r, l2, b);
    d_rad_kick<DENSE>(r, a, bp, n, k1, irho, radc, difc, bend, b);
    d_drift<DENSE>(r, l1, b);
  }
  if (h.fringe & 0xff00) quad_fringe_out(r, h, pool, s[S_B2]);
  if (bend)
    d_edge(r, (h.edge >> 8) & 0xff, irho, s[S_FX_OUT], s[S_FY_OUT], s[S_EDGE_OUT], s[S_CORR_OUT],
           -1.0, (h.flags & F_EDGEB_OUT) != 0, b);
}

__global__ void __launch_bounds__(64) diffusion_kernel(DiffArgs args) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= args.nelem) return;
  cDevElem& h = ((cDevElem*)args.elems)[e];
  double b[36];
#pragma unroll
  for (int i = 0; i < 36; i++) b[i] = 0.0;
  if (h.kind == K_STRRAD || h.kind == K_BNDRAD || h.kind == K_EXMPOLERAD) {
    const double* o = args.orbits + 6 * (int64_t)e;
    R6 r = {o[0], o[1], o[2], o[3], o[4], o[5]};
    if (!__builtin_isnan(r.x)) {
      diffusion_elem<false>(r, h, (cdouble*)args.pool, b);
      bool fine = true;
#pragma unroll
      for (int i = 0; i < 36; i++) fine = fine && __builtin_isfinite(b[i]);
      if (!fine) {
#pragma unroll
        for (int i = 0; i < 36; i++) b[i] = 0.0;
        diffusion_elem<true>(r, h, (cdouble*)args.pool, b);
      }
    }
  }
  double* out = args.bdiff + 36 * (int64_t)e;
#pragma unroll
  for (int i = 0; i < 36; i++) out[i] = b[args.row_major ? 6 * (i % 6) + i / 6 : i];
}

#endif  // ATX_AUX

// The kinds other than thick multipoles, each out of line as well.
template <int KIND>
__device__ __noinline__ R6 misc_call(R6 r, cDevElem* hp, cdouble* poolp, int nturnp) {
  cDevElem& h = *uniform(hp);
  cdouble* pool = uniform(poolp);
  if (KIND == K_IDENTITY || KIND == K_DRIFT || KIND == K_EXDRIFT) {
    // IdentityPass.c:20-43, DriftPass.c:16-48, ExactDriftPass.c:15-44
    entry_xform(r, h, pool);
    apertures(r, h, pool);
    if (KIND == K_DRIFT) drift6(r, pool[h.sc + S_D_LEN]);
    if (KIND == K_EXDRIFT) {
      exact_drift(r, pool[h.sc + S_D_LEN]);
      r.ct -= pool[h.sc + S_D_LEN];
    }
    if (KIND != K_IDENTITY) apertures(r, h, pool);
    exit_xform(r, h, pool);
  }
  if (KIND == K_THIN) thin(r, h, pool);
  if (KIND == K_RF) rf_cavity(r, h, pool, __builtin_amdgcn_readfirstlane(nturnp));
  if (KIND == K_CORR) corrector(r, h, pool);
  if (KIND == K_CAVITY) r = cavity(r, pool + h.sc, (h.flags & F_THICK) != 0);
  if (KIND == K_EXMPOLE || KIND == K_EXMPOLERAD) exact_mpole(r, h, pool, KIND == K_EXMPOLERAD);
  return r;
}

// One particle through an element by its header.
template <int U>
__device__ __forceinline__ R6 generic_element(const R6& r, cDevElem& h, cdouble* pool, int nturn) {
  switch (h.kind) {
    case K_STR: return mpole_dispatch<false, false, U>(r, h, pool);
    case K_BND: return mpole_dispatch<true, false, U>(r, h, pool);
    case K_STRRAD: return mpole_dispatch<false, true, U>(r, h, pool);
    case K_BNDRAD: return mpole_dispatch<true, true, U>(r, h, pool);
    case K_IDENTITY: return misc_call<K_IDENTITY>(r, &h, pool, nturn);
    case K_DRIFT: return misc_call<K_DRIFT>(r, &h, pool, nturn);
    case K_THIN: return misc_call<K_THIN>(r, &h, pool, nturn);
    case K_RF: return misc_call<K_RF>(r, &h, pool, nturn);
    case K_CORR: return misc_call<K_CORR>(r, &h, pool, nturn);
    case K_APERTURE: {  // AperturePass.c:9-26
      R6 v = r;
      rect_ap(v, pool + h.rap);
      return v;
    }
    case K_CAVITY: return misc_call<K_CAVITY>(r, &h, pool, nturn);
    case K_EXDRIFT: return misc_call<K_EXDRIFT>(r, &h, pool, nturn);
    case K_EXMPOLE: return misc_call<K_EXMPOLE>(r, &h, pool, nturn);
    case K_EXMPOLERAD: return misc_call<K_EXMPOLERAD>(r, &h, pool, nturn);
    default: return r;
  }
}

// at.c:115-139 predicate: any coordinate not finite, or |r_n| > 1 for n < 5, as
// the lanes of the wave that fail it: a ballot per compare is one instruction, a
// ballot of their union takes two more. After a drift of a particle that passed
// the test before it, px, py and delta are unchanged.
__device__ __forceinline__ uint64_t lost_lanes_drift(const R6& r) {
  return __builtin_amdgcn_ballot_w64(!(__builtin_fabs(r.x) <= 1.0)) |
         __builtin_amdgcn_ballot_w64(!(__builtin_fabs(r.y) <= 1.0)) |
         __builtin_amdgcn_ballot_w64(!(__builtin_fabs(r.ct) < __builtin_inf()));
}

__device__ __forceinline__ uint64_t lost_lanes(const R6& r) {
  return lost_lanes_drift(r) | __builtin_amdgcn_ballot_w64(!(__builtin_fabs(r.px) <= 1.0)) |
         __builtin_amdgcn_ballot_w64(!(__builtin_fabs(r.py) <= 1.0)) |
         __builtin_amdgcn_ballot_w64(!(__builtin_fabs(r.dp) <= 1.0));
}

// The ends of a magnet by its header: a bend's edge and the quadrupole fringe.
__device__ __noinline__ R6 ends_call(R6 r, cDevElem* hp, cdouble* poolp, int exit) {
  cDevElem& h = *uniform(hp);
  cdouble* pool = uniform(poolp);
  cdouble* s = pool + h.sc;
  const bool bend = h.kind == K_BND || h.kind == K_BNDRAD;
  if (__builtin_amdgcn_readfirstlane(exit)) {
    if (h.fringe & 0xff00) quad_fringe_out(r, h, pool, s[S_B2]);
    if (bend)
      edge<false>(r, (h.edge >> 8) & 0xff, s[S_IRHO], s[S_FX_OUT], s[S_FY_OUT], s[S_EDGE_OUT],
                  s[S_CORR_OUT], -1.0);
  } else {
    if (bend)
      edge<false>(r, h.edge & 0xff, s[S_IRHO], s[S_FX_IN], s[S_FY_IN], s[S_EDGE_IN], s[S_CORR_IN],
                  1.0);
    if (h.fringe & 0xff) quad_fringe_in(r, h, pool, s[S_B2]);
  }
  return r;
}

// Head of a program record, read one record ahead: its flags and op, the
// index of its last element, its drift's length, its number of slices and
// leading coefficient. It holds a word of the record's next two lines, too: reading
// them brings the lines into the scalar cache. (Its first constants are read with
// the record itself.)
struct OpConsts {
  double v[8];
};
struct OpHead {
  int op, last;
  double len;
  int first, nslice;
  double lead;
  OpConsts k;
  int line1, line2;
};

__device__ __forceinline__ OpConsts op_consts(cLatOp* p) {
  OpConsts k;
#pragma unroll
  for (int i = 0; i < 8; i++) k.v[i] = p->c[i];
  return k;
}

__device__ __forceinline__ OpHead op_head(cLatOp* p) {
  return OpHead{p->op, p->last, p->len, p->first, p->nslice, p->lead, OpConsts{},
                ((cint*)p)[16], ((cint*)p)[32]};
}

// A thick multipole by its record; the misalignment is applied around it by
// the caller. CHECKED, bad: rad_kick_ang.
template <bool BEND, bool RAD, int N, int F, int P, int U, bool CHECKED, class Header, class Ahead>
__device__ __forceinline__ void mpole_op(R6* r, const OpHead& o, cdouble* c, const Header& hdr,
                                         uint64_t& bad, const Ahead& ahead) {
  cdouble* a = c + (BEND && N > 1 ? OM_POLY2 : OM_POLY);
  cdouble* b = a + (N == 0 ? 2 : N + 1);
  const int nslice = o.nslice, flags = o.op;
  const OpConsts& k = o.k;
  const double irho = BEND ? k.v[OM_IRHO] : 0.0;
  if (BEND) {
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (flags & OPF_ENDS) {
        r[q] = ends_call(r[q], hdr.elem(), hdr.pool(), 0);
      } else {
        r[q].px += r[q].x * c[OM_FX_IN];
        r[q].py -= r[q].y * c[OM_FY_IN];
      }
    }
  }
  if (RAD) {
    mpole_rad_slices<BEND, N, F, P, U, CHECKED>(r, a, b, N, nslice, o.lead, k.v[OM_L1], k.v[OM_L2],
                                                k.v[OM_K1], k.v[OM_K2], irho, k.v[OM_RADC],
                                                k.v[OM_RK1], k.v[OM_RK2], bad, ahead);
  } else {
    double nl1[P], nl2[P];
#pragma unroll
    for (int q = 0; q < P; q++) {
      const double pn = rcp_opd(r[q]);
      nl1[q] = k.v[OM_L1] * pn;
      nl2[q] = k.v[OM_L2] * pn;
    }
    mpole_slices<BEND, N, F, P, U>(r, a, b, N, nslice, o.lead, nl1, nl2, k.v[OM_K1], k.v[OM_K2], irho,
                                   ahead);
  }
  if (BEND) {
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (flags & OPF_ENDS) {
        r[q] = ends_call(r[q], hdr.elem(), hdr.pool(), 1);
      } else {
        r[q].px += r[q].x * c[OM_FX_OUT];
        r[q].py -= r[q].y * c[OM_FY_OUT];
      }
    }
  }
}

// ThinMPolePass.c:42-63 by its record.
template <int N>
__device__ __forceinline__ void thin_op(R6& r, const OpConsts& k, cdouble* c) {
  cdouble* a = c + OM_POLY;
  cdouble* b = a + N + 1;
  str_kick<N>(r, a, b, N, b[N - 1], a[N - 1], 1.0);
  const double bax = k.v[OT_BAX], bay = k.v[OT_BAY];
  r.px += bax * r.dp;
  r.py -= bay * r.dp;
  r.ct -= bax * r.x - bay * r.y;
}

__device__ __forceinline__ bool is_finite(const R6& r) {
  const double inf = __builtin_inf();
  return (__builtin_fabs(r.x) < inf) & (__builtin_fabs(r.px) < inf) & (__builtin_fabs(r.y) < inf) &
         (__builtin_fabs(r.py) < inf) & (__builtin_fabs(r.dp) < inf) & (__builtin_fabs(r.ct) < inf);
}

// Roll of both planes by the angle of (c, s): the 6x6 product of mul_r
// without its zeros, in its order of summation (that it starts from 0.0 shows
// in the sign of a zero only: fill_op).
__device__ __forceinline__ void roll(R6& r, double c, double s) {
  const double x = r.x, px = r.px;
#if ATX_STRICT
  r.x = c * x + s * r.y;
  r.px = c * px + s * r.py;
  r.y = -s * x + c * r.y;
  r.py = -s * px + c * r.py;
#else
  r.x = __builtin_fma(s, r.y, c * x);
  r.px = __builtin_fma(s, r.py, c * px);
  r.y = __builtin_fma(c, r.y, -s * x);
  r.py = __builtin_fma(c, r.py, -s * px);
#endif
}

__device__ __forceinline__ void shift(R6& r, cdouble* t) {
  r.x += t[0];
  r.px += t[1];
  r.y += t[2];
  r.py += t[3];
}

#if ATX_STRICT
// A coordinate that is not finite spreads through the zeros of the 6x6
// product, as in the reference: a wave with one takes the product. (An infinite
// x of a particle without loss record enters a magnet; others come out of one.
// The fast build runs the whole element again, op_call.)
template <class Matrix>
__device__ __forceinline__ void strict_roll(R6& r, cdouble* cs, const Matrix& m) {
  if (__builtin_expect(lost_lanes(r) != 0, 0))
    r = mul_r_v(r, m());
  else
    roll(r, cs[0], cs[1]);
}
#endif

// Where an element's header and the pool are: known, or looked up in the instance
// when they are needed, so that the loop over the records does not keep them in
// scalar registers for what is rare.
struct KnownHeader {
  cDevElem* e;
  cdouble* p;
  __device__ __forceinline__ cDevElem* elem() const { return e; }
  __device__ __forceinline__ cdouble* pool() const { return p; }
};
struct LateHeader {
  cInstance* inst;
  int index;
  __device__ __forceinline__ cInstance* late() const {
    cInstance* p = inst;
    asm volatile("" : "+s"(p));
    return p;
  }
  __device__ __forceinline__ cDevElem* elem() const { return (cDevElem*)late()->elems + index; }
  __device__ __forceinline__ cdouble* pool() const { return (cdouble*)late()->pool; }
};

// The maps before and after an element that its record holds. FULL: all of them,
// otherwise those of elements without OPF_FULL. (One test for the last three first,
// in the build without copies: 3.63 against 3.73 ms per turn for 131,072 particles of
// a misaligned ring; with copies each by itself: 2.53 against 2.70 ms, 8,191.)
template <bool FULL, bool REFS, class Header>
__device__ __forceinline__ void around_entry(R6& r, int op, cdouble* c, const Header& hdr) {
  if (FULL && (op & OPF_SCALE)) change_pref(r, c[OM_SCALE]);
  if (op & OPF_XF) {
    shift(r, c + OM_XF);
#if ATX_STRICT
    if (op & OPF_R1) strict_roll(r, c + OM_XF + 4, [&]() { return hdr.pool() + hdr.elem()->r1; });
    r.dp += c[OM_ZERO];
    r.ct += c[OM_ZERO + 1];
#else
    roll(r, c[OM_XF + 4], c[OM_XF + 5]);
#endif
  }
  if (FULL && (op & OPF_HXF)) {
    cDevElem& h = *hdr.elem();
    if (h.flags & F_T1) add_t(r, hdr.pool() + h.t1);
    if (h.flags & F_R1) r = mul_r_inl(r, hdr.pool() + h.r1);
  }
  if (REFS || (op & (OPF_RAP | OPF_EAP | OPF_FRINGE))) {
    if (op & OPF_RAP) rect_ap(r, c + OM_RAP);
    if (FULL && (op & OPF_EAP)) ellip_ap(r, c + OM_EAP);
    if (op & OPF_FRINGE) r = ends_call(r, hdr.elem(), hdr.pool(), 0);
  }
}

template <bool FULL, bool REFS, class Header>
__device__ __forceinline__ void around_exit(R6& r, int op, cdouble* c, const Header& hdr) {
  if (REFS || (op & (OPF_RAP | OPF_EAP | OPF_FRINGE))) {
    if (op & OPF_FRINGE) r = ends_call(r, hdr.elem(), hdr.pool(), 1);
    // (an element without length has one aperture; the second changes nothing)
    if (op & OPF_RAP) rect_ap(r, c + OM_RAP);
    if (FULL && (op & OPF_EAP)) ellip_ap(r, c + OM_EAP);
  }
  if (FULL && (op & OPF_HXF)) {
    cDevElem& h = *hdr.elem();
    if (h.flags & F_R2) r = mul_r_inl(r, hdr.pool() + h.r2);
    if (h.flags & F_T2) add_t(r, hdr.pool() + h.t2);
  }
  if (op & OPF_XF) {
#if ATX_STRICT
    if (op & OPF_R2) strict_roll(r, c + OM_XF + 6, [&]() { return hdr.pool() + hdr.elem()->r2; });
    r.dp += c[OM_ZERO + 2];
    r.ct += c[OM_ZERO + 3];
#else
    roll(r, c[OM_XF + 6], c[OM_XF + 7]);
#endif
    shift(r, c + OM_XF + 8);
  }
  if (FULL && (op & OPF_SCALE)) change_pref(r, c[OM_SCALE + 1]);
}

// The element of a record other than its markers and drift, for the P
// particles of a lane. CHECKED, bad: rad_kick_ang; ahead: NotAhead. FULL: with the
// kinds that have OPF_FULL.
template <int P, int U, bool CHECKED, bool FULL, bool REFS, class Header, class Turn, class Ahead>
__device__ __forceinline__ void run_op(R6* r, const OpHead& o, cLatOp* rec, const Header& hdr,
                                       const Turn& nturn, uint64_t& bad, const Ahead& ahead) {
  cdouble* c = rec->c;
  const OpConsts& k = o.k;
  const int op = o.op;
  if (op & OPF_AROUND) {
#pragma unroll
    for (int q = 0; q < P; q++) around_entry<FULL, REFS>(r[q], op, c, hdr);
  }
#define ATX_MPOLE(BEND, RAD, N, F) \
  mpole_op<BEND, RAD, N, F, P, U, CHECKED>(r, o, c, hdr, bad, ahead)
  // One bit per kind, tested in groups and in the order of how common they are:
  // a test that fails falls through, where a switch becomes a tree of five
  // levels with a taken branch at most of them. (The shift is opaque, as the
  // tests would be turned into that switch.)
  uint32_t sel;
  asm("s_lshl_b32 %0, 1, %1" : "=s"(sel) : "s"(ATX_STRICT ? op >> kStrictShift : op & 0xff) : "scc");
  auto is = [&](auto... k) { return (sel & ((1u << k) | ...)) != 0; };
#if ATX_STRICT
  constexpr int kGen = F_GENERAL;  // all coefficients, whatever the form
  auto from = [&](auto k) { return (sel >> k) != 0; };
  if (from(SK_STRRAD)) {
    if (is(SK_STRRAD + 1)) ATX_MPOLE(false, true, 1, kGen);
    else if (is(SK_BNDRAD + 1)) ATX_MPOLE(true, true, 1, kGen);
    else if (is(SK_BNDRAD)) ATX_MPOLE(true, true, 0, kGen);
    else if (!FULL || is(SK_STRRAD + 2)) ATX_MPOLE(false, true, 2, kGen);
    else if (is(SK_BNDRAD + 2)) ATX_MPOLE(true, true, 2, kGen);
    else if (is(SK_STRRAD + 3)) ATX_MPOLE(false, true, 3, kGen);
    else if (is(SK_BNDRAD + 3)) ATX_MPOLE(true, true, 3, kGen);
    else ATX_MPOLE(false, true, 0, kGen);
  } else if (from(SK_STR)) {
    if (is(SK_STR + 1)) ATX_MPOLE(false, false, 1, kGen);
    else if (is(SK_STR + 2)) ATX_MPOLE(false, false, 2, kGen);
    else if (is(SK_BND + 1)) ATX_MPOLE(true, false, 1, kGen);
    else if (is(SK_STR + 3)) ATX_MPOLE(false, false, 3, kGen);
    else if (!FULL || is(SK_BND)) ATX_MPOLE(true, false, 0, kGen);
    else if (is(SK_STR)) ATX_MPOLE(false, false, 0, kGen);
    else if (is(SK_BND + 2)) ATX_MPOLE(true, false, 2, kGen);
    else ATX_MPOLE(true, false, 3, kGen);
  } else if (is(SK_THIN2)) {
#else
  constexpr int SK_THIN3 = OP_THIN3, SK_DRIFT = OP_DRIFT, SK_MARK = OP_MARK;
  if (is(OP_STRRAD1L, OP_BNDRAD0, OP_BNDRAD1L)) {
    if (is(OP_STRRAD1L)) ATX_MPOLE(false, true, 1, F_LEAD);
    else if (is(OP_BNDRAD0)) ATX_MPOLE(true, true, 1, F_NOFIELD);
    else ATX_MPOLE(true, true, 1, F_LEAD);
  } else if (is(OP_STR1L, OP_STR2L, OP_STR2D, OP_STR3L)) {
    if (is(OP_STR1L)) ATX_MPOLE(false, false, 1, F_LEAD);
    else if (is(OP_STR2L)) ATX_MPOLE(false, false, 2, F_LEAD);
    else if (is(OP_STR2D)) ATX_MPOLE(false, false, 2, F_LEAD0);
    else ATX_MPOLE(false, false, 3, F_LEAD);
  } else if (is(OP_BND0)) {
    ATX_MPOLE(true, false, 1, F_NOFIELD);
  } else if (is(OP_BND1L)) {
    ATX_MPOLE(true, false, 1, F_LEAD);
  } else if (is(OP_THIN2)) {
#endif
#pragma unroll
    for (int q = 0; q < P; q++) thin_op<2>(r[q], k, c);
    ahead();
  } else if (is(OP_CORR)) {
    ahead(k.v[OC_XK], k.v[OC_YK], k.v[OC_LEN], k.v[OC_Q0]);
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (op & OPF_THICK) {
        const double pn = rcp_opd(r[q]);
        corrector_map(r[q], k.v[OC_XK], k.v[OC_YK], k.v[OC_Q0], k.v[OC_LEN] * pn, pn);
      } else {
        r[q].px += k.v[OC_XK];
        r[q].py += k.v[OC_YK];
      }
    }
  } else if (is(OP_APERTURE)) {  // AperturePass.c:9-26
#pragma unroll
    for (int q = 0; q < P; q++) rect_ap(r[q], k.v);
    ahead();
  } else if (is(SK_DRIFT)) {
    ahead(k.v[0]);
#pragma unroll
    for (int q = 0; q < P; q++) drift6(r[q], k.v[0]);
#if !ATX_STRICT
  } else if (is(OP_STRRAD1)) {
    ATX_MPOLE(false, true, 1, F_GENERAL);
  } else if (is(OP_STR1)) {
    ATX_MPOLE(false, false, 1, F_GENERAL);
  } else if (is(OP_STR2)) {
    ATX_MPOLE(false, false, 2, F_GENERAL);
  } else if (is(OP_STR3)) {
    ATX_MPOLE(false, false, 3, F_GENERAL);
  } else if (is(OP_BNDRAD1)) {
    ATX_MPOLE(true, true, 1, F_GENERAL);
  } else if (is(OP_BND1)) {
    ATX_MPOLE(true, false, 1, F_GENERAL);
  } else if (FULL && is(OP_STRRAD2, OP_STRRAD3)) {
    if (is(OP_STRRAD2)) ATX_MPOLE(false, true, 2, F_GENERAL);
    else ATX_MPOLE(false, true, 3, F_GENERAL);
  } else if (FULL && is(OP_BNDRAD2, OP_BNDRAD3)) {
    if (is(OP_BNDRAD2)) ATX_MPOLE(true, true, 2, F_GENERAL);
    else ATX_MPOLE(true, true, 3, F_GENERAL);
  } else if (FULL && is(OP_BND2, OP_BND3)) {
    if (is(OP_BND2)) ATX_MPOLE(true, false, 2, F_GENERAL);
    else ATX_MPOLE(true, false, 3, F_GENERAL);
#endif
  } else if (is(SK_THIN3)) {
#pragma unroll
    for (int q = 0; q < P; q++) thin_op<3>(r[q], k, c);
    ahead();
  } else {
    ahead();
    if (!is(SK_MARK)) {
#pragma unroll
      for (int q = 0; q < P; q++) r[q] = generic_element<U>(r[q], *hdr.elem(), hdr.pool(), nturn());
    }
  }
#undef ATX_MPOLE
  if (op & OPF_AROUND) {
#pragma unroll
    for (int q = 0; q < P; q++) around_exit<FULL, REFS>(r[q], op, c, hdr);
  }
}

#if !ATX_STRICT
// The same out of line for one particle, with the checks in the kicks. A
// result that is not finite is computed again from the header: there a
// coordinate that is not finite spreads through the zeros of the misalignment
// matrices and of the multipole coefficients, as in the reference.
template <int U>
__device__ __noinline__ R6 op_call(R6 r, const LatOp* recp, cDevElem* hp, cdouble* poolp, int nturnp) {
  cLatOp* rec = uniform((cLatOp*)recp);
  cDevElem* h = uniform(hp);
  cdouble* pool = uniform(poolp);
  const int nturn = __builtin_amdgcn_readfirstlane(nturnp);
  R6 v = r;
  uint64_t bad = 0;
  OpHead head = op_head(rec);
  head.k = op_consts(rec);
  run_op<1, 1, true, true, false>(&v, head, rec, KnownHeader{h, pool}, [&]() { return nturn; }, bad,
                           NotAhead());
  if (rec->op & OPF_MPOLE) {
    const bool inf = !is_finite(v);
    if (__builtin_amdgcn_ballot_w64(inf) != 0) {
      const R6 g = generic_element<U>(r, *h, pool, nturn);
      v = inf ? g : v;
    }
  }
  return v;
}
#endif

// The same out of line, for the few elements of a call that are not run by
// records.
template <int U>
__device__ __noinline__ R6 header_call(R6 r, cDevElem* hp, cdouble* poolp, int nturnp) {
  return generic_element<U>(r, *uniform(hp), uniform(poolp),
                            __builtin_amdgcn_readfirstlane(nturnp));
}

__device__ __forceinline__ void store6(double* base, int64_t cs, const R6& r) {
  base[0] = r.x;
  base[cs] = r.px;
  base[2 * cs] = r.y;
  base[3 * cs] = r.py;
  base[4 * cs] = r.dp;
  base[5 * cs] = r.ct;
}

// Dynamic LDS of a workgroup of G particle slots, used to compact surviving
// particles into the leading lanes: 6*G doubles of state, G ints of particle
// index (bit 31: loss already recorded), 2 x 8 per-wave counts
// (double-buffered by round, so that a wave can publish its next count while
// a slower wave still reads the current ones).
__host__ __device__ constexpr size_t compact_lds_bytes(int slots) {
  return (size_t)slots * (6 * sizeof(double) + sizeof(int)) + 2 * 8 * sizeof(int);
}

__device__ __forceinline__ void store_state(cInstance& I, int p, const R6& r) {
  double* rp = I.r + (int64_t)p * I.pstride;
  const int64_t cs = I.cstride;
  rp[0] = r.x;
  rp[cs] = r.px;
  rp[2 * cs] = r.y;
  rp[3 * cs] = r.py;
  rp[4 * cs] = r.dp;
  rp[5 * cs] = r.ct;
}

__device__ __forceinline__ R6 load_state(cInstance& I, int p) {
  const double* rp = I.r + (int64_t)p * I.pstride;
  const int64_t cs = I.cstride;
  return R6{rp[0], rp[cs], rp[2 * cs], rp[3 * cs], rp[4 * cs], rp[5 * cs]};
}

__device__ __forceinline__ R6 lost_state() { return R6{__builtin_nan(""), 0.0, 0.0, 0.0, 0.0, 0.0}; }

// What a lane without a live particle tracks: the origin.
__device__ __forceinline__ R6 idle_state() { return R6{0.0, 0.0, 0.0, 0.0, 0.0, 0.0}; }

// A particle with its lane's state: what the loss handling changes.
struct Lane {
  R6 r;
  int flags;
};
enum : int { L_HAS = 1, L_ALIVE = 2, L_LOST = 4 };

// at.c:115-161 for the lanes with `fail` set: live particles that fail the
// loss test after element e, or whose x is NaN. Rare, so out of line, and
// called by the whole wave, so that the loop over the records has no
// divergent branch; the lane's state goes through memory, so that the loop's
// registers are not arranged around this call. A particle whose state is final is stored and its lane
// idles from then on. elempass: a NaN input of a single element pass, which
// leaves it in memory as it is.
__device__ __noinline__ void loss_call(Lane* lp, const Instance* inst, int p, int fail, int nturn,
                                       int e) {
  cInstance& I = *uniform((cInstance*)inst);
  Lane l = *lp;
  if (fail) {
    bool final = false;
    R6 fin = l.r;
    if (I.elempass) {
      final = true;
    } else if (I.losses) {
      if (!(l.flags & L_LOST)) {
        I.lost_flag[p] = 1;
        I.lost_turn[p] = (uint32_t)nturn;
        I.lost_elem[p] = (uint32_t)e;
        store6(I.lost_coord + 6 * (int64_t)p, 1, l.r);
        l.flags |= L_LOST;
        fin = lost_state();
        final = true;
      } else {
        final = __builtin_isnan(l.r.x);  // recorded by an earlier call: left as it is
      }
    } else if (__builtin_isfinite(l.r.x)) {
      fin = lost_state();
      final = true;
    } else {
      final = __builtin_isnan(l.r.x);
    }
    if (final) {
      store_state(I, p, fin);
      l.flags &= ~L_ALIVE;
      l.r = idle_state();
    }
  }
  *lp = l;
}

// Waits here for a state that a rare path has read from memory. The compiler
// would wait at the next use that the common path shares, and there for the copies
// of the record before, too (strict build, a copy at every element, 8,191
// particles: 7.17 -> 6.72 ms per turn of the large ring, with the word of copies
// waited for where it is read; no faster in the fast build).
__device__ __forceinline__ void arrived(R6& r, int& flags) {
#if ATX_STRICT
  asm volatile("" : "+v"(r.x), "+v"(r.px), "+v"(r.y), "+v"(r.py), "+v"(r.dp), "+v"(r.ct), "+v"(flags));
#endif
}

// Refpt copy: dst is the particle's six doubles in r_out; a particle whose
// state is final is copied from memory.
__device__ __noinline__ void copy_call(R6 r, const Instance* inst, double* dst, int p, int flags) {
  cInstance& I = *uniform((cInstance*)inst);
  if (flags & L_HAS) {
    if (!(flags & L_ALIVE)) r = load_state(I, p);
    store6(dst, 1, r);
  }
}

// One turn (or the part of it from e0 to e1) of a wave's particles. A function
// of its own, called once per turn: the loop over the records then has the
// scalar registers to itself instead of sharing them with everything that
// the kernel keeps for the turn boundaries.
template <int P>
struct Slots {
  Lane l[P];
  int at;  // record to go on from; kTurn: from the start, kDone: the turn is over
};
enum : int { kTurn = -1, kDone = -2 };

// FULL: with the kinds that have OPF_FULL, which cost the others registers.
// CHECKED: with the checks in the kicks of radiating magnets (fast build).
template <bool REFS, int P, int U, bool FULL, bool CHECKED>
__device__ __noinline__ Slots<P> run_turn(Slots<P> S, int p0, int p1, const Instance* instp, int tp) {
  const Instance* inst = uniform(instp);
  cInstance& I = *(cInstance*)inst;
  const int t = __builtin_amdgcn_readfirstlane(tp);
  cLatOp* ops = (cLatOp*)I.ops;
  // What is needed rarely is read from the instance again, so that the fast
  // build's loop does not keep it in scalar registers. (The strict build, whose
  // loop is larger, is 2 % faster with it kept.)
  auto late = [&]() -> cInstance& {
    cInstance* i = (cInstance*)inst;
#if !ATX_STRICT
    asm volatile("" : "+s"(i));
#endif
    return *i;
  };
  auto opof = [&](int e) { return ((cint*)late().opof)[e]; };
  const int p[2] = {p0, p1};
  R6 r[P];
  int fl[P];
#pragma unroll
  for (int q = 0; q < P; q++) {
    r[q] = S.l[q].r;
    fl[q] = S.l[q].flags;
  }
  const bool check = !I.elempass;
  auto nturn = [&]() { return late().turn0 + t; };
  const int e0 = (t == 0) ? I.start_elem : 0;
  const int e1 = I.end_elem;
  // Live particles that fail the loss test after element e: `lost` is the
  // test's result for every lane, and the lanes with a live particle are a
  // scalar mask, so that the test ends in one scalar branch.
  uint64_t alive[P];
#pragma unroll
  for (int q = 0; q < P; q++) alive[q] = __builtin_amdgcn_ballot_w64((fl[q] & L_ALIVE) != 0);
  // Refpt copy of the state before element e (at.c:622-626). The elements with
  // a copy are bits, 32 to a word, so that a word is loaded once in 32
  // elements, and the copies of a turn lie one behind the other: a rank looked
  // up per element made each element wait for a scalar load, and the copy was a
  // call. One particle with a copy at each of 320 elements took 337 us per
  // turn that way, against 189 us without copies.
  const int64_t copy = 6 * (int64_t)I.npart;
  double* dst[P];
  int word = -1;
  uint32_t here = 0;
  if (REFS) {
    const int64_t base = (t == 0) ? 0 : (int64_t)I.n_first + (int64_t)(t - 1) * I.n_std;
#pragma unroll
    for (int q = 0; q < P; q++) dst[q] = I.rout + base * copy + 6 * (int64_t)p[q];
  }
  auto copy_refs = [&](int e) {
    if ((e >> 5) != word) {
      word = e >> 5;
      cInstance& J = late();
      here = (uint32_t)((cint*)J.slots)[((t == 0) ? 0 : J.nelem / 32 + 1) + word];
#if ATX_STRICT
      asm volatile("" : "+s"(here));  // arrived()
#endif
    }
    if (!((here >> (e & 31)) & 1)) return;
#pragma unroll
    for (int q = 0; q < P; q++) {
      // A whole wave of live particles is stored without looking at its lanes
      // (8,191 particles of the large ring: 2.52 -> 2.46 ms per turn, 64: 2.32 -> 2.25).
      if (alive[q] == ~(uint64_t)0) {
        store6(dst[q], 1, r[q]);
        dst[q] += copy;
        continue;
      }
      const bool has = (fl[q] & L_HAS) != 0;
      if (__builtin_expect((__builtin_amdgcn_ballot_w64(has) & ~alive[q]) != 0, 0))
        copy_call(r[q], inst, dst[q], p[q], fl[q]);
      else if (has)
        store6(dst[q], 1, r[q]);
      dst[q] += copy;
    }
  };
  auto lose_mask = [&](int q, uint64_t bad, int e) {
    if (__builtin_expect(bad != 0, 0)) {
      Lane l{r[q], fl[q]};
      loss_call(&l, inst, p[q], (int)((bad >> (threadIdx.x & 63)) & 1), nturn(), e);
      r[q] = l.r;
      fl[q] = l.flags;
      if (REFS) arrived(r[q], fl[q]);
      alive[q] = __builtin_amdgcn_ballot_w64((fl[q] & L_ALIVE) != 0);
    }
  };
  // One element outside the loop over the records, with its refpt copy and loss
  // test. A NaN input is skipped by the first element and lost at its test.
  auto by_header = [&](int e, bool entry) {
    if (REFS) copy_refs(e);
    const LateHeader hdr{&I, e};
#pragma unroll
    for (int q = 0; q < P; q++) {
      if (entry) lose_mask(q, __builtin_amdgcn_ballot_w64(__builtin_isnan(r[q].x)) & alive[q], e);
#if !ATX_STRICT
      // in the record's form, so that a turn split into calls rounds alike
      cLatOp* rec = ops + opof(e);
      if (rec->last == e && (rec->op & OPF_MPOLE))
        r[q] = op_call<U>(r[q], (const LatOp*)rec, hdr.elem(), hdr.pool(), nturn());
      else
#endif
        r[q] = header_call<U>(r[q], hdr.elem(), hdr.pool(), nturn());
      if (check) lose_mask(q, lost_lanes(r[q]) & alive[q], e);
    }
  };
  // The loop over the records. With few waves per SIMD it was bound by the
  // time around an element's arithmetic: scalar loads waited for one after
  // the other (kind, then flags, then pool offsets, then constants), a tree of
  // branches over 147 KB of code, and the state copied for lanes that skip
  // an element. One record per drift-and-element pair with its constants at
  // fixed offsets, its head read one record ahead, no skipping lanes, tests of
  // one bit, one rare path per record, and kicks by form: the large ring (10
  // slices per magnet) from 3.35 to 1.85 ms per turn for one wave, from 3.54 to
  // 1.92 for 24,001 particles, from 8.32 to 6.25 for 262,144; the FODO ring (320
  // elements) for one wave from 354 to 162 us. What bounds it now: one wave
  // issues an FP64 instruction in 4.6 to 7.5 cycles, depending on how many of
  // its chains are independent, and four waves share the VALU's 4 cycles.
  // A turn runs the records o0..o1-1 whole. The first element of a call
  // (whose input has not passed a loss test yet) and the elements of a
  // record that a partial turn starts or ends in run by their headers,
  // before and after the records.
  const int o1 = opof(e1);
  const int from = __builtin_amdgcn_readfirstlane(S.at);
  int o0 = from >= 0 ? from : e0 < e1 ? 0 : o1;
  int e = e0;
  if (t == 0 && e0 < e1 && from < 0) {
    o0 = opof(e0) + 1;
    for (const int stop = min(ops[o0].first, e1); e < stop; e++) by_header(e, e == e0);
  }
  [[maybe_unused]] int slow = 0;  // with copies: OPF_RAD once a radiating magnet had to be run again
  cLatOp* rec = ops + o0;
  cLatOp* const end = ops + max(o0, o1);
  OpHead nxt = op_head(rec);
  for (; rec != end; rec++) {
    OpHead cur = nxt;
    asm volatile("" ::"s"(cur.line1), "s"(cur.line2));
    // The first constants are asked for here and not with the head: 16 scalar
    // registers less over the record before (24,001 particles: 2.02 against 2.05 ms
    // per turn; with a copy at every element, 8,191 particles: 2.59 against 2.74).
    cur.k = op_consts(rec);
#if ATX_STRICT
    // The strict build's divisions take long enough for the head to come, and
    // it is 6 % faster with the head asked for here (large ring, 32,003
    // particles: 7.07 against 7.55 ms per turn).
    nxt = op_head(rec + 1);
    const NotAhead ahead;
#else
    // The next record's head, asked for when this record's constants have
    // arrived: scalar loads return in any order, so that waiting for one waits
    // for all, and a constant asked for after the head would wait for the L2.
    auto ahead = [&](auto... c) {
      (hold(c), ...);
      cLatOp* p = rec + 1;
      asm volatile("" : "+s"(p));
      nxt = op_head(p);
    };
#endif
    const int kind = cur.op & 0xff;
    if (REFS) {  // markers change nothing: only their copies
      const int ndo = (kind != OP_NONE ? 1 : 0) + ((cur.op & OPF_DRIFT) ? 1 : 0);
      for (int k = cur.first; k <= cur.last - ndo; k++) copy_refs(k);
    }
    const int at = cur.last - (kind != OP_NONE ? 1 : 0);  // the drift
    // In the fast build without copies the particles that the drift lost are
    // handled with those that the element lost, the rest of the wave then takes
    // the element again: one branch to a rare path per record.
    constexpr bool kLater = !ATX_STRICT && !REFS;
    uint64_t gone[P] = {};
    if (cur.op & OPF_DRIFT) {
      if (REFS) copy_refs(at);
#pragma unroll
      for (int q = 0; q < P; q++) drift6(r[q], cur.len);
#pragma unroll
      for (int q = 0; q < P; q++) {
        gone[q] = lost_lanes_drift(r[q]) & alive[q];
        if (!kLater) lose_mask(q, gone[q], at);
      }
    }
    if (kind == OP_NONE) {
      ahead();
      if (kLater)
#pragma unroll
        for (int q = 0; q < P; q++) lose_mask(q, gone[q], at);
      continue;
    }
    if (REFS) copy_refs(cur.last);
    const LateHeader hdr{&I, cur.last};
    uint64_t bad = 0;
#if ATX_STRICT
    run_op<P, U, true, FULL, REFS>(r, cur, rec, hdr, nturn, bad, ahead);
#pragma unroll
    for (int q = 0; q < P; q++) lose_mask(q, lost_lanes(r[q]) & alive[q], cur.last);
#else
    R6 r0[P];
#pragma unroll
    for (int q = 0; q < P; q++) r0[q] = r[q];
    bool again = REFS && (cur.op & slow) != 0;
    if (REFS && __builtin_expect(again, 0)) {
      ahead();
    } else {
      run_op<P, U, CHECKED, FULL, REFS>(r, cur, rec, hdr, nturn, bad, ahead);
      again = (bad & (alive[0] | alive[P - 1])) != 0;
      if (REFS) slow |= again ? OPF_RAD : 0;
    }
    uint64_t rare = 0;
#pragma unroll
    for (int q = 0; q < P; q++) rare |= (lost_lanes(r[q]) & alive[q]) | (kLater ? gone[q] : 0);
    if (__builtin_expect(again || rare != 0, 0)) {
#pragma unroll
      for (int q = 0; q < P; q++) {
        const bool first = kLater && gone[q] != 0;
        if (first) {
          r[q] = r0[q];
          lose_mask(q, gone[q], at);
          r0[q] = r[q];
        }
        if (first || again || (cur.op & OPF_MPOLE))
          r[q] = op_call<U>(r0[q], (const LatOp*)rec, hdr.elem(), hdr.pool(), nturn());
        lose_mask(q, lost_lanes(r[q]) & alive[q], cur.last);
      }
      // Once a radiating magnet had to be run again with the checks in its kicks, the
      // wave takes the rest of the turn with the checks: a particle above 10 mrad or a
      // ring that radiates more than 2e-6 in a kick seldom has one such magnet only
      // (run again one by one, 262,144 particles of the large ring at 20 GeV took 11.7
      // ms per turn, 9.5 this way). With copies they are run one by one: the way out
      // of the loop costs it 4 %.
      if (!CHECKED && !REFS && again) {
        e = ~(int)(rec + 1 - (cLatOp*)late().ops);
        break;
      }
    }
#endif
  }
#pragma unroll
  for (int q = 0; q < P; q++) S.l[q] = Lane{r[q], fl[q]};
  S.at = kDone;
  if (!CHECKED && !REFS && e < 0) {
    S.at = ~e;
    return S;
  }
  const int stop = late().end_elem;
  for (e = max(e, ((cLatOp*)late().ops)[opof(stop)].first); e < stop; e++) by_header(e, false);
  if (REFS) copy_refs(I.nelem);
#pragma unroll
  for (int q = 0; q < P; q++) S.l[q] = Lane{r[q], fl[q]};
  return S;
}

// P particles per lane, lane-major: lane l of a workgroup holds its slots
// l*P .. l*P+P-1. live_begin (repacked turn blocks after the first; NULL
// otherwise): first workgroup of each instance among the workgroups that
// hold survivors, with live_begin[ninst] their total and live_begin[ninst +
// 1] the particle slots per workgroup (blockDim.x * P, or 64 * P when few
// survive), so that the live workgroups of all instances are the leading
// ones of the grid and the hardware spreads them evenly over the CUs; the
// other workgroups end at once.
template <bool REFS, int P, int U>
__global__ void __launch_bounds__(512, P == 1 ? 4 : 2) track_kernel(const Instance* __restrict__ insts_g, int ninst,
                                                    int nblocks, int xcd_order,
                                                    const int32_t* __restrict__ live_begin) {
  static_assert(P == 1 || P == 2, "one or two particles per lane");
  extern __shared__ double lds[];
  cInstance* insts = (cInstance*)insts_g;
  // Workgroup order (xcd_order: a launch over several instances of equal
  // turn counts): the hardware deals workgroup i to XCD i mod kXcds, and
  // each XCD has its own L2. The workgroups of the launch (nblocks, or the
  // live ones of a repacked turn block) are dealt in kXcds contiguous
  // chunks, one per XCD, so that the instances (lattices) of one chunk are
  // read through one L2 rather than every L2 holding every lattice. The
  // grid is kXcds * ceil(nblocks / kXcds) workgroups; the first kXcds *
  // ceil(nlog / kXcds) of them map one to one onto the logical workgroups
  // below that count, and those past nlog, like the rest, end at once. The
  // hardware order stands otherwise: one lattice is read alike by every
  // XCD, and items of unequal turn counts, dealt in chunks, would load the
  // XCDs unevenly.
  const int nlog = live_begin ? live_begin[ninst] : nblocks;
  const int hw = (int)blockIdx.x;
  int bid = hw;
  if (xcd_order) {
    const int chunk = (nlog + kXcds - 1) / kXcds;
    if (hw >= kXcds * chunk) return;
    bid = (hw % kXcds) * chunk + hw / kXcds;
  }
  if (bid >= nlog) return;
  // Instance of this workgroup: the last whose first block is <= bid.
  int lo = 0, hi = ninst - 1;
  int wbegin;
  int G = (int)blockDim.x * P;  // particle slots per workgroup
  if (live_begin) {
    G = live_begin[ninst + 1];
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (live_begin[mid] <= bid) lo = mid; else hi = mid - 1;
    }
    wbegin = live_begin[lo];
  } else {
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (insts[mid].block_begin <= bid) lo = mid; else hi = mid - 1;
    }
    wbegin = insts[lo].block_begin;
  }
  cInstance& I = insts[lo];
  const int tid = (int)threadIdx.x;
  const int npart = I.npart;
  // lanes of a repacked launch take the surviving particles idx[0..nlive)
  const int32_t* idx = I.idx;
  const int nslot = idx ? __builtin_amdgcn_readfirstlane(*I.nlive) : npart;
  const int first = (bid - wbegin) * G;  // first slot of this workgroup
  // particles of this workgroup, and its waves that hold some (uniform);
  // the other waves end now
  int held = max(0, min(G, nslot - first));
  int nw = (held + 64 * P - 1) / (64 * P);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wave >= nw) return;

  const int losses = I.losses;
  int p[P];
  // Of each slot: whether it holds a particle (L_HAS), whether the
  // particle's state is in the lane's registers (L_ALIVE), and whether its
  // loss has been recorded (L_LOST). A particle whose x is NaN is skipped by
  // every element (at.c:142-161, *Pass.c): its state goes to memory for good
  // when it is found (at the loss test, or at the first element for a NaN
  // input) and the lane tracks the origin from then on, so that no element
  // needs to mask lanes or keep their old state.
  Lane L[P];
#pragma unroll
  for (int q = 0; q < P; q++) {
    const int sl = tid * P + q;
    const bool has = sl < held;
    p[q] = has ? (idx ? idx[first + sl] : first + sl) : 0;
    L[q].r = idle_state();
    L[q].flags = L_LOST;  // a slot without a particle never records a loss
    if (has) {
      L[q].r = load_state(I, p[q]);
      L[q].flags = L_HAS | L_ALIVE;
      if (losses == 2) {
        if (I.lost_flag[p[q]] != 0) L[q].flags |= L_LOST;  // recorded by an earlier call
      } else if (losses) {
        I.lost_flag[p[q]] = 0;
        I.lost_turn[p[q]] = 0;
        I.lost_elem[p[q]] = 0;
        store6(I.lost_coord + 6 * (int64_t)p[q], 1, R6{0.0, 0.0, 0.0, 0.0, 0.0, 0.0});
      }
    }
  }

  const bool check = !I.elempass;
  const int nturns = I.nturns;
  // Lost particles are dropped at turn boundaries and the survivors packed
  // into the leading lanes: with one particle per lane when packing frees a
  // wave (the waves left without particles end and free their SIMD slots),
  // with several whenever one was lost (a lane steps its particles together
  // only while none of them is lost). Not with refpts: lost particles still
  // fill their refpt copies, as in at.c.
  const bool ends = !REFS && (I.n_first | I.n_std) != 0;  // copies at the end of a turn only
  const bool compact = check && !REFS && !ends && nturns > 1;
  double* s_r = lds;
  int* s_p = (int*)(lds + 6 * G);
  int* s_cnt = s_p + G;
  for (int t = 0; t < nturns; t++) {
    if (compact && t > 0) {
      // drop the particles whose final state is stored
      int mine = 0, below = 0;
      int within[P];
#pragma unroll
      for (int q = 0; q < P; q++) {
        const bool on = (L[q].flags & L_ALIVE) != 0;
        const uint64_t m = __builtin_amdgcn_ballot_w64(on);
        within[q] = mine;
        mine += on ? 1 : 0;
        below += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                           __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
      }
      int cnt = mine;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
      int* cnt_buf = s_cnt + 8 * (t & 1);
      if ((tid & 63) == 0) cnt_buf[wave] = cnt;
      __syncthreads();
      int off = 0, total = 0;
      for (int k = 0; k < nw; k++) {
        const int c = cnt_buf[k];
        off += (k < wave) ? c : 0;
        total += c;
      }
      total = __builtin_amdgcn_readfirstlane(total);
      const int need = (total + 64 * P - 1) / (64 * P);
      if (need < nw || (P > 1 && total < held)) {  // uniform
#pragma unroll
        for (int q = 0; q < P; q++) {
          if (L[q].flags & L_ALIVE) {
            const int j = off + below + within[q];
            s_r[j] = L[q].r.x;
            s_r[G + j] = L[q].r.px;
            s_r[2 * G + j] = L[q].r.y;
            s_r[3 * G + j] = L[q].r.py;
            s_r[4 * G + j] = L[q].r.dp;
            s_r[5 * G + j] = L[q].r.ct;
            s_p[j] = p[q] | ((L[q].flags & L_LOST) ? (int)0x80000000u : 0);
          }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < P; q++) {
          const int j = tid * P + q;
          if (j < total) {
            L[q].r.x = s_r[j];
            L[q].r.px = s_r[G + j];
            L[q].r.y = s_r[2 * G + j];
            L[q].r.py = s_r[3 * G + j];
            L[q].r.dp = s_r[4 * G + j];
            L[q].r.ct = s_r[5 * G + j];
            const int v = s_p[j];
            p[q] = v & 0x7fffffff;
            L[q].flags = L_HAS | L_ALIVE | (v < 0 ? L_LOST : 0);
          } else {
            L[q].flags = L_LOST;
          }
        }
        held = total;
        nw = need;
        if (wave >= nw) return;  // this wave holds no particle any more
      }
    }
#pragma unroll
    for (int q = 0; q < P; q++)
      if (!(L[q].flags & L_ALIVE)) L[q].r = idle_state();
    Slots<P> S;
#pragma unroll
    for (int q = 0; q < P; q++) S.l[q] = L[q];
    S.at = kTurn;
    if (I.full)
      S = run_turn<REFS, P, U, true, ATX_STRICT>(S, p[0], p[P - 1], insts_g + lo, t);
    else
      S = run_turn<REFS, P, U, false, ATX_STRICT>(S, p[0], p[P - 1], insts_g + lo, t);
    if (!ATX_STRICT && !REFS && __builtin_amdgcn_readfirstlane(S.at) >= 0)
      S = run_turn<REFS, P, U, true, true>(S, p[0], p[P - 1], insts_g + lo, t);
#pragma unroll
    for (int q = 0; q < P; q++) L[q] = S.l[q];
    if (ends) {
      const int64_t base = (t == 0) ? 0 : (int64_t)I.n_first + (int64_t)(t - 1) * I.n_std;
      double* out = I.rout + base * 6 * (int64_t)npart;
#pragma unroll
      for (int q = 0; q < P; q++) {
        if (!(L[q].flags & L_HAS)) continue;
        const bool alive = (L[q].flags & L_ALIVE) != 0;
        store6(out + 6 * (int64_t)p[q], 1, alive ? L[q].r : load_state(I, p[q]));
      }
    }
  }
#pragma unroll
  for (int q = 0; q < P; q++)
    if (L[q].flags & L_ALIVE) store_state(I, p[q], L[q].r);
}

}  // namespace ATX_NS
}  // namespace atx

// The kernel of this object's launch shape: nblocks workgroups of `block`
// lanes, block * ATX_PPT particle slots each.
extern "C" hipError_t ATX_LAUNCH(const atx::Instance* d_insts, int ninst, int nblocks, int block,
                                 int refs, int xcd_order, const int32_t* live_begin,
                                 hipStream_t stream) {
  const size_t lds = atx::ATX_NS::compact_lds_bytes(block * ATX_PPT);
  // whole rounds of XCDs: the kernel's workgroup order needs the grid to
  // cover kXcds * ceil(n / kXcds) for every n <= nblocks
  const int grid = (nblocks + atx::kXcds - 1) / atx::kXcds * atx::kXcds;
  if (refs)
    hipLaunchKernelGGL((atx::ATX_NS::track_kernel<true, ATX_PPT, ATX_UNROLL>), dim3(grid),
                       dim3(block), lds, stream, d_insts, ninst, nblocks, xcd_order, live_begin);
  else
    hipLaunchKernelGGL((atx::ATX_NS::track_kernel<false, ATX_PPT, ATX_UNROLL>), dim3(grid),
                       dim3(block), lds, stream, d_insts, ninst, nblocks, xcd_order, live_begin);
  return hipGetLastError();
}

#if ATX_PPT == 1 && ATX_UNROLL == (ATX_STRICT ? 1 : 2)
namespace atx {
namespace ATX_NS {
// Element matrices (matrix.py:195-202): lane c of element e's wave tracks its
// entrance orbit plus column c of [D, -D], D = diag(step/2), through element e
// alone (at.c at_elempass: no loss test, a NaN input stays as it is); the zeros
// of -D are -0.0, as numpy adds them. m[i][j] = (probe j+ - probe j-)_i / step,
// column-major or row-major, each column written by its lane.
// One kernel from orbits to matrices: as a batch of single-element launches
// this took a 448 KB instance table from the host and two kernels around the
// tracking one. A wave per element keeps the element's constants scalar; the
// idle lanes cost nothing, the launch (2,241 elements of a large ring: 2.2
// waves per SIMD) is as long as the chain of one magnet. The bounds are those of
// the tracking kernel, whose functions it calls.
__global__ void __launch_bounds__(512, 4) element_matrix_kernel(ElemMatArgs args) {
  const int e = (int)blockIdx.x;
  const int c = (int)threadIdx.x;
  const double h = 0.5 * args.step;
  const double* o = args.orbits + 6 * (int64_t)e;
  const double d = (c < 6) ? h : -h;
  const double z = (c < 6) ? 0.0 : -0.0;
  const int k = c % 6;
  R6 r = {o[0] + (k == 0 ? d : z), o[1] + (k == 1 ? d : z), o[2] + (k == 2 ? d : z),
          o[3] + (k == 3 ? d : z), o[4] + (k == 4 ? d : z), o[5] + (k == 5 ? d : z)};
  const R6 in = r;
  const bool skip = __builtin_isnan(r.x);
  if (skip || c >= 12) r = idle_state();
  cDevElem* h_e = (cDevElem*)args.elems + e;
#if !ATX_STRICT
  cLatOp* rec = (cLatOp*)args.ops + ((cint*)args.opof)[e];
  if (rec->last == e && (rec->op & OPF_MPOLE))
    r = op_call<ATX_UNROLL>(r, (const LatOp*)rec, h_e, (cdouble*)args.pool, 1);
  else
#endif
    r = header_call<ATX_UNROLL>(r, h_e, (cdouble*)args.pool, 1);
  if (skip) r = in;
  const double v[6] = {r.x, r.px, r.y, r.py, r.dp, r.ct};
  const int row = args.row_major ? 6 : 1, col = args.row_major ? 1 : 6;
  double* m = args.m66 + 36 * (int64_t)e + col * c;
#pragma unroll
  for (int i = 0; i < 6; i++) {
    const double minus = __shfl_down(v[i], 6, 64);
    if (c < 6) m[row * i] = (v[i] - minus) / args.step;
  }
}
}  // namespace ATX_NS
}  // namespace atx

#if ATX_STRICT
#define ATX_LAUNCH_ELEM atx_launch_element_matrices_strict
#else
#define ATX_LAUNCH_ELEM atx_launch_element_matrices_fast
#endif
extern "C" hipError_t ATX_LAUNCH_ELEM(const atx::ElemMatArgs* args, hipStream_t stream) {
  if (args->nelem <= 0) return hipSuccess;
  hipLaunchKernelGGL(atx::ATX_NS::element_matrix_kernel, dim3((unsigned)args->nelem), dim3(64), 0,
                     stream, *args);
  return hipGetLastError();
}
#endif

#if ATX_AUX
namespace atx {
// Repack between the turn blocks of a batched launch: one workgroup per
// instance lists, in order, the particles still alive (x not NaN: a lost
// particle is set to NaN, at.c:142-161) in idx[0..*nlive). The first pass
// scans 0..npart, later passes the previous list, in place: a chunk is read
// completely before it is written, and writes never pass the read front.
__global__ void __launch_bounds__(1024) repack_kernel(const Instance* __restrict__ insts,
                                                      int first_pass) {
  __shared__ int s_wave[16];
  const Instance& I = insts[blockIdx.x];
  int32_t* idx = const_cast<int32_t*>(I.idx);
  int32_t* nlive = const_cast<int32_t*>(I.nlive);
  if (!idx) return;
  const int n = first_pass ? I.npart : *nlive;
  const int tid = (int)threadIdx.x;
  const int wave = tid >> 6;
  const int nwaves = (int)blockDim.x >> 6;
  int out = 0;
  for (int base = 0; base < n; base += (int)blockDim.x) {
    const int s = base + tid;
    int q = 0;
    bool alive = false;
    if (s < n) {
      q = first_pass ? s : idx[s];
      alive = !__builtin_isnan(I.r[(int64_t)q * I.pstride]);
    }
    const uint64_t m = __builtin_amdgcn_ballot_w64(alive);
    const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                               __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
    if ((tid & 63) == 0) s_wave[wave] = __popcll(m);
    __syncthreads();
    int off = 0, total = 0;
    for (int k = 0; k < nwaves; k++) {
      const int c = s_wave[k];
      off += (k < wave) ? c : 0;
      total += c;
    }
    if (alive) idx[out + off + rank] = q;
    out += total;
    __syncthreads();
  }
  if (tid == 0) *nlive = out;
}
}  // namespace atx

namespace atx {
// Live particles of instance i with turns in the block (0 for the others).
__device__ __forceinline__ int live_count(const Instance& I) {
  return I.nturns > 0 ? (I.idx ? *I.nlive : I.npart) : 0;
}

// Map of the live workgroups for the next turn block (one workgroup):
// live_begin[i] = sum over j < i of ceil(nlive_j / g), live_begin[ninst] =
// the total and live_begin[ninst + 1] = g, the particles per workgroup: the
// block size, or 64 when all survivors fit in fine_limit lanes (then each
// workgroup runs one wave and the dispatcher spreads single waves over the
// SIMDs, which a tail of few survivors needs; the grid holds enough
// workgroups for either). Chunks of 1,024 instances: a wave-level scan, then
// the wave totals through LDS, carrying the running sum from chunk to chunk.
__global__ void __launch_bounds__(1024) live_map_kernel(const Instance* __restrict__ insts, int ninst,
                                                        int block, int fine, int fine_limit,
                                                        int32_t* __restrict__ live_begin) {
  __shared__ int s_wave[16];
  __shared__ int s_total;
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int nwaves = (int)blockDim.x >> 6;
  // total survivors
  int part = 0;
  for (int i = tid; i < ninst; i += (int)blockDim.x) part += live_count(insts[i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
  if (lane == 0) s_wave[wave] = part;
  __syncthreads();
  if (tid == 0) {
    int t = 0;
    for (int k = 0; k < nwaves; k++) t += s_wave[k];
    s_total = t;
  }
  __syncthreads();
  const int g = s_total <= fine_limit ? fine : block;
  int carry = 0;
  for (int base = 0; base < ninst; base += (int)blockDim.x) {
    const int i = base + tid;
    int c = 0;
    if (i < ninst) c = (live_count(insts[i]) + g - 1) / g;
    int v = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int u = __shfl_up(v, off, 64);
      if (lane >= off) v += u;
    }
    if (lane == 63) s_wave[wave] = v;
    __syncthreads();
    int woff = 0, total = 0;
    for (int k = 0; k < nwaves; k++) {
      const int w = s_wave[k];
      woff += (k < wave) ? w : 0;
      total += w;
    }
    if (i < ninst) live_begin[i] = carry + woff + v - c;
    carry += total;
    __syncthreads();
  }
  if (tid == 0) {
    live_begin[ninst] = carry;
    live_begin[ninst + 1] = g;
  }
}
}  // namespace atx

extern "C" hipError_t atx_launch_repack(const atx::Instance* d_insts, int ninst, int first_pass,
                                        hipStream_t stream) {
  if (ninst <= 0) return hipSuccess;
  hipLaunchKernelGGL(atx::repack_kernel, dim3(ninst), dim3(1024), 0, stream, d_insts, first_pass);
  return hipGetLastError();
}

extern "C" hipError_t atx_launch_live_map(const atx::Instance* d_insts, int ninst, int block,
                                          int fine, int fine_limit, int32_t* live_begin,
                                          hipStream_t stream) {
  if (ninst <= 0) return hipSuccess;
  hipLaunchKernelGGL(atx::live_map_kernel, dim3(1), dim3(1024), 0, stream, d_insts, ninst, block,
                     fine, fine_limit, live_begin);
  return hipGetLastError();
}

extern "C" hipError_t atx_launch_diffusion(const atx::DiffArgs* args, hipStream_t stream) {
  const int block = 64;
  const int nblocks = (args->nelem + block - 1) / block;
  if (nblocks == 0) return hipSuccess;
  hipLaunchKernelGGL(atx::ATX_NS::diffusion_kernel, dim3(nblocks), dim3(block), 0, stream, *args);
  return hipGetLastError();
}
#endif
