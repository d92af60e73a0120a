// atx_adjoint.hip -- reverse-mode (adjoint) kernel of the tracking map.
//
// Gradient of a loss of the final particle coordinates with respect to the
// state at the start of a block of turns and to the multipole coefficients
// PolynomB[k] of selected elements. One lane per particle walks the turns of
// the block backwards and, inside each turn, the elements and their
// Forest-Ruth sub-steps in reverse order. The input state of every sub-step
// is reconstructed by inverting that sub-step exactly in closed form (every
// map of the supported pass methods is a shear: drift, thin kick, edge
// kick, RF energy kick, corrector, misalignment), starting each turn from
// the exact turn-start state recorded by the forward tracking kernel, so no
// per-element storage is needed and reconstruction error never spans more
// than one turn. The adjoint uses the transposed per-step Jacobians of the
// reference tangent maps (diff_drift.c:2-28, diff_thinkick.c:1-35,
// diff_bnd_kick.c:1-46, edge terms of diff_bend_fringe.c:32-48).
#include <hip/hip_runtime.h>

#include "atx_device.h"
#include "atx_libm.h"

namespace atx {
namespace adj {

typedef __attribute__((address_space(4))) const double cdouble;
typedef __attribute__((address_space(4))) const DevElem cDevElem;
typedef __attribute__((address_space(4))) const AdjElem cAdjElem;
typedef __attribute__((address_space(4))) const AdjItem cAdjItem;
typedef __attribute__((address_space(4))) const LatOp cLatOp;
typedef __attribute__((address_space(4))) const AdjRec cAdjRec;
typedef __attribute__((address_space(4))) const int32_t cint;

struct V6 {
  double x, px, y, py, dp, ct;
};

// 1/d within an ulp: the hardware estimate and two Newton steps.
__device__ __forceinline__ double rcp(double d) {
  double q = __builtin_amdgcn_rcp(d);
  q = __builtin_fma(q, __builtin_fma(-d, q, 1.0), q);
  return __builtin_fma(q, __builtin_fma(-d, q, 1.0), q);
}

// polynomial value and complex derivative: sum (B_k + i A_k) z^k, z = x + i y
template <int N>
__device__ __forceinline__ void field_d(double x, double y, cdouble* a, cdouble* b, int n,
                                        double& re, double& im, double& ren, double& imn) {
  const int order = (N >= 0) ? N : n;
  re = b[order];
  im = a[order];
  ren = 0.0;
  imn = 0.0;
#pragma unroll
  for (int k = order - 1; k >= 0; k--) {
    const double tr = ren * x - imn * y + re;
    imn = ren * y + imn * x + im;
    ren = tr;
    const double t = re * x - im * y + b[k];
    im = re * y + im * x + a[k];
    re = t;
  }
}

// Re, Im of z^j for the coefficient gradient
__device__ __forceinline__ void zpow(double x, double y, int j, double& zr, double& zi) {
  zr = 1.0;
  zi = 0.0;
  for (int i = 0; i < j; i++) {
    const double t = zr * x - zi * y;
    zi = zr * y + zi * x;
    zr = t;
  }
}

// Reverse of an in-magnet drift x' = x + nl px, ct' = ct + nl (px^2+py^2) u/2
// with nl = L u, u = 1/(1+dp).
__device__ __forceinline__ void drift_rev(V6& r, V6& l, double len) {
  const double u = rcp(1.0 + r.dp);
  const double nl = len * u;
  const double p2 = r.px * r.px + r.py * r.py;
  r.x -= nl * r.px;
  r.y -= nl * r.py;
  r.ct -= nl * p2 * 0.5 * u;
  const double nlu = nl * u;
  l.dp -= nlu * (r.px * l.x + r.py * l.y + p2 * u * l.ct);
  l.px += nl * l.x + nlu * r.px * l.ct;
  l.py += nl * l.y + nlu * r.py * l.ct;
}

// Reverse of a thin multipole kick of integrated length k (straight or
// curved frame). g accumulates dL/dB_jg.
template <bool BEND, int N>
__device__ __forceinline__ void kick_rev(V6& r, V6& l, cdouble* a, cdouble* b, int n, double k,
                                         double h, int jg, double& g) {
  double re, im, ren, imn;
  field_d<N>(r.x, r.y, a, b, n, re, im, ren, imn);
  if (jg >= 0) {
    double zr, zi;
    zpow(r.x, r.y, jg, zr, zi);
    g += k * (zi * l.py - zr * l.px);
  }
  const double lx = -k * ren * l.px + k * imn * l.py;
  const double ly = k * imn * l.px + k * ren * l.py;
  if (BEND) {
    l.x += lx - k * h * h * l.px + k * h * l.ct;
    l.dp += k * h * l.px;
    r.px += k * (re - (r.dp - r.x * h) * h);
    r.ct -= k * h * r.x;
  } else {
    l.x += lx;
    r.px += k * re;
  }
  l.y += ly;
  r.py -= k * im;
}

// v plus the v of the lane that the DPP control names (0 where there is none):
// moves between lanes inside the VALU, where a shuffle goes through the LDS unit
// and its latency.
template <int CTRL>
__device__ __forceinline__ double plus_dpp(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
  return v + __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Sum of the wave in lane 63: within rows of 16 lanes (shifts right by 1, 2, 4,
// 8), then each row's last lane to the next row, then to the upper half.
__device__ __forceinline__ void grad_flush(double g, int slot, double* grad) {
  g = plus_dpp<0x111>(g);
  g = plus_dpp<0x112>(g);
  g = plus_dpp<0x114>(g);
  g = plus_dpp<0x118>(g);
  g = plus_dpp<0x142>(g);
  g = plus_dpp<0x143>(g);
  if ((threadIdx.x & 63) == 63) atomicAdd(grad + slot, g);
}

// misalignment: state r <- Minv r, adjoint l <- M^T l
__device__ __noinline__ void mat_rev(V6& r, V6& l, cdouble* m, cdouble* minv) {
  const double v[6] = {r.x, r.px, r.y, r.py, r.dp, r.ct};
  const double w[6] = {l.x, l.px, l.y, l.py, l.dp, l.ct};
  double o[6], q[6];
  for (int i = 0; i < 6; i++) {
    double s = 0.0, t = 0.0;
    for (int j = 0; j < 6; j++) {
      s += minv[i + 6 * j] * v[j];
      t += m[j + 6 * i] * w[j];
    }
    o[i] = s;
    q[i] = t;
  }
  r = V6{o[0], o[1], o[2], o[3], o[4], o[5]};
  l = V6{q[0], q[1], q[2], q[3], q[4], q[5]};
}

__device__ __forceinline__ void sub_t(V6& r, cdouble* t) {
  r.x -= t[0];
  r.px -= t[1];
  r.y -= t[2];
  r.py -= t[3];
  r.dp -= t[4];
  r.ct -= t[5];
}

__device__ __forceinline__ void exit_rev(V6& r, V6& l, cDevElem& h, cAdjElem& ae, cdouble* pool) {
  if (h.flags & F_T2) sub_t(r, pool + h.t2);
  if (h.flags & F_R2) mat_rev(r, l, pool + h.r2, pool + ae.r2inv);
}

__device__ __forceinline__ void entry_rev(V6& r, V6& l, cDevElem& h, cAdjElem& ae, cdouble* pool) {
  if (h.flags & F_R1) mat_rev(r, l, pool + h.r1, pool + ae.r1inv);
  if (h.flags & F_T1) sub_t(r, pool + h.t1);
}

// edge kick px' = px + x fx, py' = py - y fy (E_CONST) or fy = c0/(1+dp) (E_DIVP)
__device__ __forceinline__ void edge_rev(V6& r, V6& l, int mode, double fx, double c0) {
  const double u = 1.0 / (1.0 + r.dp);
  const double fy = (mode == E_DIVP) ? c0 * u : c0;
  if (mode == E_DIVP) l.dp += r.y * c0 * u * u * l.py;
  l.x += fx * l.px;
  l.y -= fy * l.py;
  r.px -= r.x * fx;
  r.py += r.y * fy;
}

template <bool BEND, int N>
__device__ __forceinline__ void mpole_rev(V6& r, V6& l, cDevElem& h, cAdjElem& ae, cdouble* pool,
                                          double* grad) {
  cdouble* s = pool + h.sc;
  cdouble* a = pool + h.poly;
  cdouble* b = a + h.order + 1;
  const int n = h.order;
  const int jg = (ae.slot >= 0 && grad) ? ae.coeff : -1;
  double g = 0.0;
  const double irho = s[S_IRHO];
  exit_rev(r, l, h, ae, pool);
  if (BEND) edge_rev(r, l, (h.edge >> 8) & 0xff, s[S_FX_OUT], s[S_FY_OUT]);
  const double l1 = s[S_L1], l2 = s[S_L2], k1 = s[S_K1], k2 = s[S_K2];
  for (int m = 0; m < h.nslice; m++) {
    drift_rev(r, l, l1);
    kick_rev<BEND, N>(r, l, a, b, n, k1, irho, jg, g);
    drift_rev(r, l, l2);
    kick_rev<BEND, N>(r, l, a, b, n, k2, irho, jg, g);
    drift_rev(r, l, l2);
    kick_rev<BEND, N>(r, l, a, b, n, k1, irho, jg, g);
    drift_rev(r, l, l1);
  }
  if (BEND) edge_rev(r, l, h.edge & 0xff, s[S_FX_IN], s[S_FY_IN]);
  entry_rev(r, l, h, ae, pool);
  if (jg >= 0) grad_flush(g, ae.slot, grad);
}

template <bool BEND>
__device__ __forceinline__ void mpole_rev_dispatch(V6& r, V6& l, cDevElem& h, cAdjElem& ae,
                                                   cdouble* pool, double* grad) {
  switch (h.order) {
    case 1: mpole_rev<BEND, 1>(r, l, h, ae, pool, grad); break;
    case 2: mpole_rev<BEND, 2>(r, l, h, ae, pool, grad); break;
    case 3: mpole_rev<BEND, 3>(r, l, h, ae, pool, grad); break;
    default: mpole_rev<BEND, -1>(r, l, h, ae, pool, grad); break;
  }
}

__device__ __forceinline__ void thin_rev(V6& r, V6& l, cDevElem& h, cAdjElem& ae, cdouble* pool,
                                         double* grad) {
  cdouble* s = pool + h.sc;
  cdouble* a = pool + h.poly;
  cdouble* b = a + h.order + 1;
  const int jg = (ae.slot >= 0 && grad) ? ae.coeff : -1;
  double g = 0.0;
  exit_rev(r, l, h, ae, pool);
  const double bax = s[S_BAX], bay = s[S_BAY];
  // ct' = ct - bax x + bay y; px' = px + bax dp; py' = py - bay dp
  r.ct += bax * r.x - bay * r.y;
  r.px -= bax * r.dp;
  r.py += bay * r.dp;
  l.x -= bax * l.ct;
  l.y += bay * l.ct;
  l.dp += bax * l.px - bay * l.py;
  kick_rev<false, -1>(r, l, a, b, h.order, 1.0, 0.0, jg, g);
  entry_rev(r, l, h, ae, pool);
  if (jg >= 0) grad_flush(g, ae.slot, grad);
}

// full drift with its own 1/(1+dp): same Jacobian as drift_rev
__device__ __forceinline__ void rf_rev(V6& r, V6& l, cDevElem& h, cdouble* pool, int nturn) {
  cdouble* s = pool + h.sc;
  const double nt = (double)nturn;
  if (h.flags & F_THICK) drift_rev(r, l, s[S_RF_HALF]);
  if (h.flags & F_RFKICK) {
    const double tw = s[S_RF_TWOPIF];
    double ph, sn;
    {
      // the forward kick's phase and sine, bit for bit, so the inverse is exact
#pragma clang fp contract(off)
      ph = tw * ((r.ct - s[S_RF_LAG]) / 2.99792458e8 - s[S_RF_HFT0] * nt) - s[S_RF_PHILAG];
      sn = libm::host_sin(ph);
    }
    const double cs = cos(ph);
    r.dp += s[S_RF_NV] * sn;  // undo dp += -nv sin(ph)
    l.ct += -s[S_RF_NV] * cs * tw / 2.99792458e8 * l.dp;
  }
  if (h.flags & F_THICK) drift_rev(r, l, s[S_RF_HALF]);
}

__device__ __forceinline__ void corrector_rev(V6& r, V6& l, cDevElem& h, cAdjElem& ae,
                                              cdouble* pool) {
  cdouble* s = pool + h.sc;
  const double xk = s[S_C_XK], yk = s[S_C_YK];
  exit_rev(r, l, h, ae, pool);
  r.px -= xk;
  r.py -= yk;
  if (h.flags & F_THICK) {
    // forward (from the input state): ct += nl u Q/2, x += nl (px + xk/2),
    // y += nl (py + yk/2), with nl = L u, u = 1/(1+dp)
    const double u = 1.0 / (1.0 + r.dp);
    const double nl = s[S_C_LEN] * u;
    r.x -= nl * (r.px + 0.5 * xk);
    r.y -= nl * (r.py + 0.5 * yk);
    const double q = xk * xk / 3.0 + yk * yk / 3.0 + r.px * r.px + r.py * r.py + r.px * xk + r.py * yk;
    r.ct -= nl * u * q * 0.5;
    const double nlu = nl * u;
    l.dp -= nlu * ((r.px + 0.5 * xk) * l.x + (r.py + 0.5 * yk) * l.y + q * u * l.ct);
    l.px += nl * l.x + nlu * (r.px + 0.5 * xk) * l.ct;
    l.py += nl * l.y + nlu * (r.py + 0.5 * yk) * l.ct;
  }
  entry_rev(r, l, h, ae, pool);
}

__device__ __forceinline__ void element_rev(V6& r, V6& l, cDevElem& h, cAdjElem& ae, cdouble* pool,
                                            double* grad, int nturn) {
  switch (h.kind) {
    case K_IDENTITY:
      exit_rev(r, l, h, ae, pool);
      entry_rev(r, l, h, ae, pool);
      break;
    case K_DRIFT:
      exit_rev(r, l, h, ae, pool);
      drift_rev(r, l, pool[h.sc + S_D_LEN]);
      entry_rev(r, l, h, ae, pool);
      break;
    case K_STR: mpole_rev_dispatch<false>(r, l, h, ae, pool, grad); break;
    case K_BND: mpole_rev_dispatch<true>(r, l, h, ae, pool, grad); break;
    case K_THIN: thin_rev(r, l, h, ae, pool, grad); break;
    case K_RF: rf_rev(r, l, h, pool, nturn); break;
    case K_CORR: corrector_rev(r, l, h, ae, pool); break;
    default: break;  // AperturePass: identity for surviving particles
  }
}

// --- Elements by their records -----------------------------------------------
// Reverse of the ops that a ring without radiation is made of. In a magnet
// delta and lambda_ct are constant, so the reciprocal 1/(1+delta) and every
// product of a drift's length with them are taken once per magnet: a drift is
// 13 FP64 instructions instead of 35 (a division among them), two drifts in a
// row are one, and the kicks are spelled out for the form of the field (7
// instead of about 20 for a quadrupole). 4,096 particles and 8 turns of the large
// ring: the two sweeps 21.0 -> 9.6 ms.
struct RevDrift {
  double nl, nlu;     // L u, L u^2 with u = 1/(1+delta)
  double hh;          // L u^2 / 2
  double d, c;        // L u^2 lambda_ct, L u^3 lambda_ct
};

__device__ __forceinline__ RevDrift rev_drift(double len, double u, double lct) {
  RevDrift k;
  k.nl = len * u;
  k.nlu = k.nl * u;
  k.hh = 0.5 * k.nlu;
  k.d = k.nlu * lct;
  k.c = k.d * u;
  return k;
}

__device__ __forceinline__ void drift_rev(V6& r, V6& l, const RevDrift& k) {
  const double p2 = __builtin_fma(r.px, r.px, r.py * r.py);
  const double t = __builtin_fma(r.px, l.x, r.py * l.y);
  r.x = __builtin_fma(-k.nl, r.px, r.x);
  r.y = __builtin_fma(-k.nl, r.py, r.y);
  r.ct = __builtin_fma(-k.hh, p2, r.ct);
  l.dp = __builtin_fma(-k.nlu, t, __builtin_fma(-k.c, p2, l.dp));
  l.px = __builtin_fma(k.nl, l.x, __builtin_fma(k.d, r.px, l.px));
  l.py = __builtin_fma(k.nl, l.y, __builtin_fma(k.d, r.py, l.py));
}

struct RevKick {
  double kl, kb, kb2;    // length, length times B[N], twice that
  double kh, khh, khl;   // bends: length times curvature, its square, lambda_ct
  double bn, bn2;        // DIPOLE: B[N], twice that, B[0], A[0]
  double b0, a0;
};

// Kick of length kl of a field B[N] z^N (LEAD) or none, in a straight or curved
// frame; DIPOLE: with B[0] and A[0]; GRAD: g += d lambda / d B[N].
template <bool BEND, int N, bool LEAD, bool DIPOLE, bool GRAD>
__device__ __forceinline__ void kick_rev(V6& r, V6& l, const RevKick& k, double irho, double& g) {
  static_assert(!DIPOLE || (LEAD && N == 2), "a sextupole that is a corrector, too");
  const double x = r.x, y = r.y, lx = l.px, ly = l.py;
  if (BEND) {
    r.px = __builtin_fma(-k.kh, __builtin_fma(-x, irho, r.dp), r.px);
    r.ct = __builtin_fma(-k.kh, x, r.ct);
    l.x = __builtin_fma(-k.khh, lx, l.x + k.khl);
    l.dp = __builtin_fma(k.kh, lx, l.dp);
  }
  if (!LEAD) return;
  const double s = __builtin_fma(y, ly, -x * lx);  // y l_py - x l_px
  if (N == 1) {
    r.px = __builtin_fma(k.kb, x, r.px);
    r.py = __builtin_fma(-k.kb, y, r.py);
    l.x = __builtin_fma(-k.kb, lx, l.x);
    l.y = __builtin_fma(k.kb, ly, l.y);
    if (GRAD) g = __builtin_fma(k.kl, s, g);
  } else {
    const double t = __builtin_fma(y, lx, x * ly);  // y l_px + x l_py
    const double zr = __builtin_fma(x, x, -(y * y)), zi = 2.0 * x * y;
    if (N == 2) {
      if (DIPOLE) {
        r.px = __builtin_fma(k.kl, __builtin_fma(k.bn, zr, k.b0), r.px);
        r.py = __builtin_fma(-k.kl, __builtin_fma(k.bn2, x * y, k.a0), r.py);
      } else {
        r.px = __builtin_fma(k.kb, zr, r.px);
        r.py = __builtin_fma(-k.kb, zi, r.py);
      }
      l.x = __builtin_fma(k.kb2, s, l.x);
      l.y = __builtin_fma(k.kb2, t, l.y);
      if (GRAD) g = __builtin_fma(k.kl, __builtin_fma(zi, ly, -zr * lx), g);
    } else {  // z^3 = zr x - zi y + i (zr y + zi x); derivative 3 z^2
      const double cr = __builtin_fma(zr, x, -zi * y), ci = __builtin_fma(zr, y, zi * x);
      const double k3 = 3.0 * k.kb;
      r.px = __builtin_fma(k.kb, cr, r.px);
      r.py = __builtin_fma(-k.kb, ci, r.py);
      l.x = __builtin_fma(k3, __builtin_fma(zi, ly, -zr * lx), l.x);
      l.y = __builtin_fma(k3, __builtin_fma(zi, lx, zr * ly), l.y);
      if (GRAD) g = __builtin_fma(k.kl, __builtin_fma(ci, ly, -cr * lx), g);
    }
  }
}

__device__ __forceinline__ void hold(double v) { asm volatile("" ::"s"(v)); }

// ahead: asks for the next record, called when this one's constants have
// arrived (scalar loads return in any order: a wait for one waits for all).
template <bool BEND, int N, bool LEAD, bool DIPOLE, bool GRAD, class Ahead>
__device__ __forceinline__ double mpole_rev_op(V6& r, V6& l, cdouble* c, int nslice, double lead,
                                               const Ahead& ahead) {
  const double bn = LEAD ? lead : 0.0;
  double b0 = 0.0, a0 = 0.0;
  if (DIPOLE) {
    a0 = c[OM_POLY];
    b0 = c[OM_POLY + N + 1];
    asm("" : "=v"(a0) : "0"(a0));  // an FMA reads one scalar
    asm("" : "=v"(b0) : "0"(b0));
  }
  hold(c[OM_L1]);
  hold(c[OM_L2]);
  hold(c[OM_K1]);
  hold(c[OM_K2]);
  if (LEAD) hold(bn);
  if (BEND) hold(c[OM_FX_OUT]);
  ahead();
  const double irho = BEND ? c[OM_IRHO] : 0.0;
  const double u = rcp(1.0 + r.dp);
  const RevDrift d1 = rev_drift(c[OM_L1], u, l.ct), d2 = rev_drift(c[OM_L2], u, l.ct);
  const RevDrift d11 = {2.0 * d1.nl, 2.0 * d1.nlu, 2.0 * d1.hh, 2.0 * d1.d, 2.0 * d1.c};
  RevKick k[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    k[i].kl = c[OM_K1 + i];
    k[i].kb = k[i].kl * bn;
    k[i].kb2 = 2.0 * k[i].kb;
    k[i].kh = k[i].kl * irho;
    k[i].khh = k[i].kh * irho;
    k[i].khl = k[i].kh * l.ct;
    k[i].bn = bn;
    k[i].bn2 = 2.0 * bn;
    k[i].b0 = b0;
    k[i].a0 = a0;
  }
  double g = 0.0;
  if (BEND) {
    const double fx = c[OM_FX_OUT], fy = c[OM_FY_OUT];
    l.x = __builtin_fma(fx, l.px, l.x);
    l.y = __builtin_fma(-fy, l.py, l.y);
    r.px = __builtin_fma(-r.x, fx, r.px);
    r.py = __builtin_fma(r.y, fy, r.py);
  }
  auto body = [&]() {
    kick_rev<BEND, N, LEAD, DIPOLE, GRAD>(r, l, k[0], irho, g);
    drift_rev(r, l, d2);
    kick_rev<BEND, N, LEAD, DIPOLE, GRAD>(r, l, k[1], irho, g);
    drift_rev(r, l, d2);
    kick_rev<BEND, N, LEAD, DIPOLE, GRAD>(r, l, k[0], irho, g);
  };
  if (nslice > 0) {
    drift_rev(r, l, d1);
    for (int m = 1; m < nslice; m++) {
      body();
      drift_rev(r, l, d11);
    }
    body();
    drift_rev(r, l, d1);
  }
  if (BEND) {
    const double fx = c[OM_FX_IN], fy = c[OM_FY_IN];
    l.x = __builtin_fma(fx, l.px, l.x);
    l.y = __builtin_fma(-fy, l.py, l.y);
    r.px = __builtin_fma(-r.x, fx, r.px);
    r.py = __builtin_fma(r.y, fy, r.py);
  }
  return g;
}

template <bool BEND, int N, bool LEAD, bool DIPOLE, class Ahead>
__device__ __forceinline__ void mpole_rev_rec(V6& r, V6& l, cdouble* c, int nslice, double lead,
                                              int slot, double* grad, const Ahead& ahead) {
  if (LEAD && slot >= 0 && grad)
    grad_flush(mpole_rev_op<BEND, N, LEAD, DIPOLE, true>(r, l, c, nslice, lead, ahead), slot, grad);
  else
    mpole_rev_op<BEND, N, LEAD, DIPOLE, false>(r, l, c, nslice, lead, ahead);
}

// A roll of both planes: x' = c x + s y, y' = -s x + c y, and (ci, si) its
// inverse's: r <- R^-1 r, l <- R^T l.
__device__ __forceinline__ void roll_rev(V6& r, V6& l, double c, double s, double ci, double si) {
  const double x = r.x, px = r.px, lx = l.x, lpx = l.px;
  r.x = __builtin_fma(-si, r.y, ci * x);
  r.px = __builtin_fma(-si, r.py, ci * px);
  r.y = __builtin_fma(ci, r.y, si * x);
  r.py = __builtin_fma(ci, r.py, si * px);
  l.x = __builtin_fma(-s, l.y, c * lx);
  l.px = __builtin_fma(-s, l.py, c * lpx);
  l.y = __builtin_fma(c, l.y, s * lx);
  l.py = __builtin_fma(c, l.py, s * lpx);
}

__device__ __forceinline__ void shift_rev(V6& r, cdouble* t) {
  r.x -= t[0];
  r.px -= t[1];
  r.y -= t[2];
  r.py -= t[3];
}

// grid: x over the particles of the largest item, y over the items; lanes
// beyond an item's particle count idle with zero adjoint (a workgroup with
// none of its particles returns at once: the kernel has no barrier)
__global__ void __launch_bounds__(256, 2) adjoint_kernel(AdjArgs args) {
  cAdjItem& it = ((cAdjItem*)args.items)[blockIdx.y];
  const int npart = it.npart;
  if ((int)(blockIdx.x * blockDim.x) >= npart) return;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  const bool active = p < npart;
  const int64_t np6 = 6 * (int64_t)npart;
  const double* states = it.states;
  double* grad = it.grad;
  cDevElem* elems = (cDevElem*)args.elems;
  cAdjElem* aes = (cAdjElem*)args.adj;
  cdouble* pool = (cdouble*)args.pool;
  // inactive lanes (beyond N, or particles lost by the end of the block)
  // run with zero adjoint so that every lane reaches the wave reductions
  const double* send = states + (int64_t)it.nturns * np6 + 6 * (int64_t)(active ? p : 0);
  bool live = active && __builtin_isfinite(send[0]);
  V6 l = {0, 0, 0, 0, 0, 0};
  if (live) {
    const double* lp = it.lam + 6 * (int64_t)p;
    l = V6{lp[0], lp[1], lp[2], lp[3], lp[4], lp[5]};
  }
  for (int t = it.nturns - 1; t >= 0; t--) {
    const double* sp = states + (int64_t)(t + 1) * np6 + 6 * (int64_t)(active ? p : 0);
    V6 r = {0, 0, 0, 0, 0, 0};
    if (live) r = V6{sp[0], sp[1], sp[2], sp[3], sp[4], sp[5]};
    const int nturn = it.turn0 + t;
    // the records backwards: their element, then their drift; markers change
    // nothing
    cLatOp* rec = (cLatOp*)args.ops + (args.nops - 1);
    cAdjRec* ar = (cAdjRec*)args.recs + (args.nops - 1);
    struct Head {
      int op, last;
      double len;
      int nslice, slot, coeff, line1;
    };
    auto head = [](cLatOp* p, cAdjRec* q) {
      return Head{p->op, p->last, p->len, p->nslice, q->slot, q->coeff, ((cint*)p)[16]};
    };
    Head nxt{0, 0, 0.0, 0, -1, 0, 0};
    if (args.nops > 0) nxt = head(rec, ar);
    for (int i = args.nops - 1; i >= 0; i--, rec--, ar--) {
      const Head cur = nxt;
      asm volatile("" ::"s"(cur.line1));
      const int kind = cur.op & 0xff, sl = cur.slot;
      cdouble* c = rec->c;
      auto ahead = [&]() {
        if (i == 0) return;
        cLatOp* p = rec - 1;
        asm volatile("" : "+s"(p));
        nxt = head(p, ar - 1);
      };
      // the record's form, unless its gradient is of another coefficient or its
      // edges are in the header
      const int order = kind == OP_STR2L || kind == OP_STR2D ? 2 : kind == OP_STR3L ? 3 : 1;
      const bool form = kind >= OP_STR1L && kind <= OP_BND0 && !(cur.op & (OPF_ENDS | OPF_HXF)) &&
                        (sl < 0 || (cur.coeff == order && kind != OP_BND0));
      const bool moved = form && (cur.op & OPF_XF);
      if (moved) {
        shift_rev(r, c + OM_XF + 8);
        roll_rev(r, l, c[OM_XF + 6], c[OM_XF + 7], c[OM_INV + 2], c[OM_INV + 3]);
      }
      switch (form ? kind : (kind == OP_NONE || kind == OP_APERTURE || kind == OP_MARK ? OP_NONE : OP_GENERIC)) {
#define ATX_REV(BEND, N, LEAD, DIPOLE) \
  mpole_rev_rec<BEND, N, LEAD, DIPOLE>(r, l, c, cur.nslice, rec->lead, sl, grad, ahead)
        case OP_NONE: ahead(); break;
        case OP_STR1L: ATX_REV(false, 1, true, false); break;
        case OP_STR2L: ATX_REV(false, 2, true, false); break;
        case OP_STR2D: ATX_REV(false, 2, true, true); break;
        case OP_STR3L: ATX_REV(false, 3, true, false); break;
        case OP_BND1L: ATX_REV(true, 1, true, false); break;
        case OP_BND0: ATX_REV(true, 1, false, false); break;
#undef ATX_REV
        default: {
          ahead();
          // Inline: as a function it costs the loop its scalar registers (9.8
          // against 8.8 ms for 8 turns of 4,096 particles of the large ring), and
          // with its pointers in vector registers the loads are one per lane (a
          // corrected error realisation without forms for misalignment: 126 ms).
          // On copies: the matrix products take the states by address, and the
          // loop's own would live in memory (12.1 ms).
          V6 r1 = r, l1 = l;
          element_rev(r1, l1, elems[cur.last], aes[cur.last], pool, grad, nturn);
          r = r1;
          l = l1;
        }
      }
      if (moved) {
        roll_rev(r, l, c[OM_XF + 4], c[OM_XF + 5], c[OM_INV], c[OM_INV + 1]);
        shift_rev(r, c + OM_XF);
      }
      if (cur.op & OPF_DRIFT) {
        const double u = rcp(1.0 + r.dp);
        drift_rev(r, l, rev_drift(cur.len, u, l.ct));
      }
    }
  }
  if (active) {
    double* lp = it.lam + 6 * (int64_t)p;
    lp[0] = l.x;
    lp[1] = l.px;
    lp[2] = l.y;
    lp[3] = l.py;
    lp[4] = l.dp;
    lp[5] = l.ct;
  }
}

}  // namespace adj
}  // namespace atx

// max_npart: the largest particle count of the items (host-side copy of the
// device item table); nitems <= 65535 (grid y limit)
extern "C" hipError_t atx_launch_adjoint(const atx::AdjArgs* args, int32_t max_npart,
                                         hipStream_t stream) {
  // Few waves run one to a workgroup, each on a CU that it shares with as few as
  // possible (4,096 particles: 2.29 ms per turn, 2.51 in workgroups of four);
  // from about two per CU on, a workgroup of four puts one on each SIMD of a
  // CU, where single ones pile up (65,536 particles: 2.8 ms, 3.6 one by one).
  // Two waves per SIMD suffice: with registers for four the sweep is 3 to 5 %
  // slower at every size from 64 to 11,000 waves.
  const int64_t waves = (int64_t)((max_npart + 63) / 64) * args->nitems;
  const int block = waves <= 512 ? 64 : 256;
  const int nblocks = (max_npart + block - 1) / block;
  if (nblocks == 0 || args->nitems <= 0) return hipSuccess;
  hipLaunchKernelGGL(atx::adj::adjoint_kernel, dim3(nblocks, args->nitems), dim3(block), 0, stream,
                     *args);
  return hipGetLastError();
}
