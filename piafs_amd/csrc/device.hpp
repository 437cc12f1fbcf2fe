// Device functions shared by the kernels: nonlinear weights and interpolation,
// the eigenstructures, the upwinders at one interface, ensemble indexing.
// Include from .hip files only; everything has internal linkage.
#pragma once

#include "kernels.hpp"

namespace piafs {

namespace {

// ---------------------------------------------------------------------------
// Quotient n / d for the WENO weights and the CRWENO5 multipliers: the
// target's IEEE double division (a reciprocal estimate, two Newton-Raphson
// refinements and one residual correction, Markstein's method) without its
// range scaling and special-case fix-up steps, in three fewer instructions
// and with no condition register between them.  Those steps are identities,
// and the result is the IEEE quotient's bits, while n is +0 or of magnitude at
// least 2^-969, d is normal and positive, and the quotient lies within
// 2^-969 .. 2^1022: for the weights, whenever the smoothness indicators stay
// within about 2^400 of epsilon (data of ordinary magnitude with the usual
// epsilons).  Far outside (epsilon 1e-100 with data of 1e70), a weight below
// about 1e-290 can differ in its last bits, and where a Z or YC ratio
// overflows the row's weights are all NaN rather than partly NaN: the
// interpolated value is still NaN as the reference's is, and a tiny weight's
// term lies far below the last bit of a sum led by the large weights.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wdiv(double n, double d) {
  const double r0 = __builtin_amdgcn_rcp(d);
  const double e0 = __builtin_fma(-d, r0, 1.0);
  const double r1 = __builtin_fma(r0, e0, r0);
  const double e1 = __builtin_fma(-d, r1, 1.0);
  const double r2 = __builtin_fma(r1, e1, r1);
  const double q = n * r2;
  const double t = __builtin_fma(-d, q, n);
  return __builtin_fma(t, r2, q);
}

// ---------------------------------------------------------------------------
// WENO5 nonlinear weights, include/interpolation.h:255-490
// (JS :255-281, mapped :309-341, Z (Borges) :420-450, YC :478-508)
// ---------------------------------------------------------------------------
// from the smoothness indicators b1..b3; t: YC's fourth difference
template <int KIND>
__device__ __forceinline__ void weno_of(double c1, double c2, double c3, double b1, double b2, double b3, double t,
                                        double eps, double &w1, double &w2, double &w3) {
  double a1, a2, a3;
  if (KIND == 2 || KIND == 3) {
    const double tau = KIND == 2 ? fabs(b3 - b1) : t * t;
    const double r1 = wdiv(tau, b1 + eps), r2 = wdiv(tau, b2 + eps), r3 = wdiv(tau, b3 + eps);
    a1 = c1 * (1.0 + r1 * r1);
    a2 = c2 * (1.0 + r2 * r2);
    a3 = c3 * (1.0 + r3 * r3);
  } else {
    a1 = wdiv(c1, (b1 + eps) * (b1 + eps));
    a2 = wdiv(c2, (b2 + eps) * (b2 + eps));
    a3 = wdiv(c3, (b3 + eps) * (b3 + eps));
  }
  double s = wdiv(1.0, a1 + a2 + a3);
  w1 = a1 * s;
  w2 = a2 * s;
  w3 = a3 * s;
  if (KIND == 1) {
    a1 = wdiv(w1 * (c1 + c1 * c1 - 3 * c1 * w1 + w1 * w1), c1 * c1 + w1 * (1.0 - 2.0 * c1));
    a2 = wdiv(w2 * (c2 + c2 * c2 - 3 * c2 * w2 + w2 * w2), c2 * c2 + w2 * (1.0 - 2.0 * c2));
    a3 = wdiv(w3 * (c3 + c3 * c3 - 3 * c3 * w3 + w3 * w3), c3 * c3 + w3 * (1.0 - 2.0 * c3));
    s = wdiv(1.0, a1 + a2 + a3);
    w1 = a1 * s;
    w2 = a2 * s;
    w3 = a3 * s;
  }
}

template <int KIND>
__device__ __forceinline__ void weno_w(double c1, double c2, double c3, double m3, double m2, double m1,
                                       double p1, double p2, double eps, double &w1, double &w2, double &w3) {
  // 2, 4 and 1/4 scale exactly, so each of those products joins its sum in one
  // fma with the same bits
  const double t1312 = 13.0 / 12.0, q14 = 1.0 / 4.0;
  const double d1 = __builtin_fma(-2.0, m2, m3) + m1, e1 = __builtin_fma(-4.0, m2, m3) + 3 * m1;
  const double d2 = __builtin_fma(-2.0, m1, m2) + p1, e2 = m2 - p1;
  const double d3 = __builtin_fma(-2.0, p1, m1) + p2, e3 = __builtin_fma(-4.0, p1, 3 * m1) + p2;
  const double b1 = __builtin_fma(q14, e1 * e1, t1312 * d1 * d1);
  const double b2 = __builtin_fma(q14, e2 * e2, t1312 * d2 * d2);
  const double b3 = __builtin_fma(q14, e3 * e3, t1312 * d3 * d3);
  const double t = KIND == 3 ? m3 - 4 * m2 + 6 * m1 - 4 * p1 + p2 : 0.0;
  weno_of<KIND>(c1, c2, c3, b1, b2, b3, t, eps, w1, w2, w3);
}

__device__ __forceinline__ void weno_w_rt(int kind, double c1, double c2, double c3, double m3, double m2,
                                          double m1, double p1, double p2, double eps, double &w1, double &w2,
                                          double &w3) {
  switch (kind) {
    case 1: weno_w<1>(c1, c2, c3, m3, m2, m1, p1, p2, eps, w1, w2, w3); break;
    case 2: weno_w<2>(c1, c2, c3, m3, m2, m1, p1, p2, eps, w1, w2, w3); break;
    case 3: weno_w<3>(c1, c2, c3, m3, m2, m1, p1, p2, eps, w1, w2, w3); break;
    default: weno_w<0>(c1, c2, c3, m3, m2, m1, p1, p2, eps, w1, w2, w3); break;
  }
}

// Candidate stencils of WENO5 (Interp1PrimFifthOrderWENO.c:151-153) and of the
// compact scheme (Interp1PrimFifthOrderCRWENO.c:176-179).
__device__ __forceinline__ void weno5_cands(double m3, double m2, double m1, double p1, double p2, double &f1,
                                            double &f2, double &f3) {
  const double s6 = 1.0 / 6.0;
  f1 = (2 * s6) * m3 + (-7 * s6) * m2 + (11 * s6) * m1;
  f2 = (-s6) * m2 + (5 * s6) * m1 + (2 * s6) * p1;
  f3 = (2 * s6) * m1 + (5 * s6) * p1 + (-s6) * p2;
}
__device__ __forceinline__ void crweno5_cands(double m2, double m1, double p1, double &f1, double &f2,
                                              double &f3) {
  const double s6 = 1.0 / 6.0;
  f1 = (s6)*m2 + (5 * s6) * m1;
  f2 = (5 * s6) * m1 + (s6)*p1;
  f3 = (s6)*m1 + (5 * s6) * p1;
}

// Linear fifth-order upwind interpolation (upw5),
// Interp1PrimFifthOrderUpwind.c:92-96 and :138-142, in the reference's
// operation order (sums left to right).
__device__ __forceinline__ double upw5_value(double m3, double m2, double m1, double p1, double p2) {
  const double c30 = 1.0 / 30.0, c13 = 13.0 / 60.0, c47 = 47.0 / 60.0, c27 = 27.0 / 60.0, c20 = 1.0 / 20.0;
  return c30 * m3 - c13 * m2 + c47 * m1 + c27 * p1 - c20 * p2;
}

// Coefficients of row k of one compact line system: A, B, C and the right-hand
// side (the end rows are identity rows carrying the WENO5 value).
template <int KIND>
__device__ __forceinline__ void row_coeffs(int k, int N, bool left, const ReconParams &R, double w0, double w1,
                                           double w2, double w3, double w4, double w5, double &Ak, double &Bk,
                                           double &Ck, double &Rk) {
  double m3, m2, m1, p1, p2;
  if (left) { m3 = w0; m2 = w1; m1 = w2; p1 = w3; p2 = w4; }
  else { m3 = w5; m2 = w4; m1 = w3; p1 = w2; p2 = w1; }
  const bool bnd = (k == 0) || (k == N);
  double c1, c2, c3;
  if (!bnd) { c1 = 0.2; c2 = 0.5; c3 = 0.3; }
  else { c1 = 0.1; c2 = 0.6; c3 = 0.3; }
  double a1, a2, a3;
  if (R.no_limiting) { a1 = c1; a2 = c2; a3 = c3; }
  else weno_w<KIND>(c1, c2, c3, m3, m2, m1, p1, p2, R.eps, a1, a2, a3);
  double f1, f2, f3;
  if (bnd) {
    weno5_cands(m3, m2, m1, p1, p2, f1, f2, f3);
    Ak = 0.0; Bk = 1.0; Ck = 0.0;
  } else {
    const double t3 = 1.0 / 3.0;
    crweno5_cands(m2, m1, p1, f1, f2, f3);
    const double lo = (2 * t3) * a1 + (t3)*a2;
    Bk = (t3)*a1 + (2 * t3) * a2 + (2 * t3) * a3;
    const double hi = (t3)*a3;
    if (left) { Ak = lo; Ck = hi; } else { Ak = hi; Ck = lo; }
  }
  Rk = a1 * f1 + a2 * f2 + a3 * f3;
}

// ---------------------------------------------------------------------------
// 1D Euler eigenstructure, euler1d.h:91-193
// ---------------------------------------------------------------------------
struct Eig3 {
  double L[3][3], R[3][3], D[3];
};

__device__ __forceinline__ void euler1d_roeavg(double g, double rhoL, double muL, double eL, double rhoR,
                                               double muR, double eR, double &r0, double &r1, double &r2) {
  const double vL = muL / rhoL, PL = (eL - 0.5 * rhoL * vL * vL) * (g - 1.0), cLsq = g * PL / rhoL;
  const double HL = 0.5 * vL * vL + cLsq / (g - 1.0);
  const double vR = muR / rhoR, PR = (eR - 0.5 * rhoR * vR * vR) * (g - 1.0), cRsq = g * PR / rhoR;
  const double HR = 0.5 * vR * vR + cRsq / (g - 1.0);
  const double tL = sqrt(rhoL), tR = sqrt(rhoR);
  const double rho = tL * tR, v = (tL * vL + tR * vR) / (tL + tR), H = (tL * HL + tR * HR) / (tL + tR);
  const double csq = (g - 1.0) * (H - 0.5 * v * v), P = csq * rho / g;
  r0 = rho;
  r1 = rho * v;
  r2 = P / (g - 1.0) + 0.5 * rho * v * v;
}

__device__ __forceinline__ void euler1d_eig(double g, double u0, double u1, double u2, Eig3 &E) {
  const double rho = u0, v = u1 / rho, e = u2;
  const double P = (e - 0.5 * rho * v * v) * (g - 1.0), c = sqrt(g * P / rho);
  E.D[0] = v; E.D[1] = v - c; E.D[2] = v + c;
  const double k = (g - 1) / (rho * c);
  E.L[1][0] = k * (-(v * v) / 2 - c * v / (g - 1));
  E.L[1][1] = k * (v + c / (g - 1));
  E.L[1][2] = k * (-1);
  E.L[0][0] = k * (rho * (-(v * v) / 2 + c * c / (g - 1)) / c);
  E.L[0][1] = k * (rho * v / c);
  E.L[0][2] = k * (-rho / c);
  E.L[2][0] = k * ((v * v) / 2 - c * v / (g - 1));
  E.L[2][1] = k * (-v + c / (g - 1));
  E.L[2][2] = k * (1);
  E.R[0][1] = -rho / (2 * c);
  E.R[1][1] = -rho * (v - c) / (2 * c);
  E.R[2][1] = -rho * ((v * v) / 2 + (c * c) / (g - 1) - c * v) / (2 * c);
  E.R[0][0] = 1; E.R[1][0] = v; E.R[2][0] = v * v / 2;
  E.R[0][2] = rho / (2 * c);
  E.R[1][2] = rho * (v + c) / (2 * c);
  E.R[2][2] = rho * ((v * v) / 2 + (c * c) / (g - 1) + c * v) / (2 * c);
}

// ---------------------------------------------------------------------------
// 2D Navier-Stokes flow eigenstructure along direction DIR (0: x, 1: y).
// Only the 4x4 flow block is formed: the species block of the reference's
// n x n matrices is the identity (L, R) with eigenvalue vn.
// ---------------------------------------------------------------------------
// Roe average of two conserved flow states (navierstokes2d.h:115-160)
__device__ __forceinline__ void ns2d_roeavg(double g, const double uL[4], const double uR[4], double ua[4]) {
  const double rhoL = uL[0], vxL = uL[1] / rhoL, vyL = uL[2] / rhoL, eL = uL[3];
  const double vsqL = (vxL * vxL) + (vyL * vyL), PL = (eL - 0.5 * rhoL * vsqL) * (g - 1.0);
  const double cLsq = g * PL / rhoL, HL = 0.5 * (vxL * vxL + vyL * vyL) + cLsq / (g - 1.0);
  const double rhoR = uR[0], vxR = uR[1] / rhoR, vyR = uR[2] / rhoR, eR = uR[3];
  const double vsqR = (vxR * vxR) + (vyR * vyR), PR = (eR - 0.5 * rhoR * vsqR) * (g - 1.0);
  const double cRsq = g * PR / rhoR, HR = 0.5 * (vxR * vxR + vyR * vyR) + cRsq / (g - 1.0);
  const double tL = sqrt(rhoL), tR = sqrt(rhoR);
  const double rA = tL * tR;
  const double vxA = (tL * vxL + tR * vxR) / (tL + tR), vyA = (tL * vyL + tR * vyR) / (tL + tR);
  const double HA = (tL * HL + tR * HR) / (tL + tR), vsqA = vxA * vxA + vyA * vyA;
  const double csqA = (g - 1.0) * (HA - 0.5 * vsqA), PA = csqA * rA / g;
  ua[0] = rA;
  ua[1] = rA * vxA;
  ua[2] = rA * vyA;
  ua[3] = PA / (g - 1.0) + 0.5 * rA * vsqA;
}

// Flow eigenvalues, in the reference's order (navierstokes2d.h:161-184)
template <int DIR>
__device__ __forceinline__ void ns2d_eigvals(double g, const double u[4], double D[4]) {
  const double rho = u[0], vx = (rho == 0) ? 0 : u[1] / rho, vy = (rho == 0) ? 0 : u[2] / rho, e = u[3];
  const double vsq = (vx * vx) + (vy * vy), P = (e - 0.5 * rho * vsq) * (g - 1.0);
  const double a = sqrt(g * P / rho), vn = DIR == 0 ? vx : vy;
  D[0] = vn - a;
  if (DIR == 0) { D[1] = vn + a; D[2] = vn; }
  else { D[1] = vn; D[2] = vn + a; }
  D[3] = vn;
}

// |v_n| of the Roe average of two cells with the Harten entropy fix
// (delta = 1e-6, NavierStokes2DUpwind.c:75-78): the species' dissipation
// coefficient of the Roe flux, as upwind_ns2d_roe computes it
template <int DIR>
__device__ __forceinline__ double ns2d_roe_dsp(double g, const double uLc[4], const double uRc[4]) {
  double ua[4], D[4];
  ns2d_roeavg(g, uLc, uRc, ua);
  ns2d_eigvals<DIR>(g, ua, D);
  const double vn = D[3];
  const double delta = 0.000001, delta2 = delta * delta;
  return fabs(vn) < delta ? (vn * vn + delta2) / (2 * delta) : fabs(vn);
}

// right flow eigenvectors (columns) from the sound speed, the velocity, the
// kinetic energy per mass and the enthalpy h0
template <int DIR>
__device__ __forceinline__ void ns2d_right(double a, double vx, double vy, double ek, double h0, double R[4][4]) {
  const double nx = DIR == 0 ? 1.0 : 0.0, ny = DIR == 0 ? 0.0 : 1.0, un = DIR == 0 ? vx : vy;
  R[0][0] = 1.0; R[1][0] = vx - a * nx; R[2][0] = vy - a * ny; R[3][0] = h0 - a * un;
  R[0][3] = 1.0; R[1][3] = vx; R[2][3] = vy; R[3][3] = ek;
  const int cp = DIR == 0 ? 1 : 2, cz = DIR == 0 ? 2 : 1;
  R[0][cp] = 1.0; R[1][cp] = vx + a * nx; R[2][cp] = vy + a * ny; R[3][cp] = h0 + a * un;
  R[0][cz] = 0.0; R[1][cz] = ny; R[2][cz] = -nx; R[3][cz] = vx * ny - vy * nx;
}

// Left (rows) and right (columns) flow eigenvectors (navierstokes2d.h:186-311);
// ns: sound speed, velocity, kinetic energy and h0, from which R follows
template <int DIR>
__device__ __forceinline__ void ns2d_left(double g, const double u[4], double L[4][4], double ns[5]) {
  const double gm1 = g - 1.0;
  const double rho = u[0], vx = (rho == 0) ? 0 : u[1] / rho, vy = (rho == 0) ? 0 : u[2] / rho, e = u[3];
  const double vsq = (vx * vx) + (vy * vy), P = (e - 0.5 * rho * vsq) * (g - 1.0);
  const double a = sqrt(g * P / rho), ek = 0.5 * (vx * vx + vy * vy);
  const double aa2 = 2 * a * a, aa = a * a;
  if (DIR == 0) {
    const double un = vx, nx = 1.0, ny = 0.0;
    L[0][0] = (gm1 * ek + a * un) / aa2;
    L[0][1] = ((-gm1) * vx - a * nx) / aa2;
    L[0][2] = ((-gm1) * vy - a * ny) / aa2;
    L[0][3] = gm1 / aa2;
    L[3][0] = (aa - gm1 * ek) / aa;
    L[3][1] = (gm1 * vx) / aa;
    L[3][2] = (gm1 * vy) / aa;
    L[3][3] = (-gm1) / aa;
    L[1][0] = (gm1 * ek - a * un) / aa2;
    L[1][1] = ((-gm1) * vx + a * nx) / aa2;
    L[1][2] = ((-gm1) * vy + a * ny) / aa2;
    L[1][3] = gm1 / aa2;
    L[2][0] = (vy - un * ny) / nx;
    L[2][1] = ny;
    L[2][2] = (ny * ny - 1.0) / nx;
    L[2][3] = 0.0;
  } else {
    const double un = vy, nx = 0.0, ny = 1.0;
    L[0][0] = (gm1 * ek + a * un) / aa2;
    L[0][1] = ((1.0 - g) * vx - a * nx) / aa2;
    L[0][2] = ((1.0 - g) * vy - a * ny) / aa2;
    L[0][3] = gm1 / aa2;
    L[3][0] = (aa - gm1 * ek) / aa;
    L[3][1] = gm1 * vx / aa;
    L[3][2] = gm1 * vy / aa;
    L[3][3] = (1.0 - g) / aa;
    L[2][0] = (gm1 * ek - a * un) / aa2;
    L[2][1] = ((1.0 - g) * vx + a * nx) / aa2;
    L[2][2] = ((1.0 - g) * vy + a * ny) / aa2;
    L[2][3] = gm1 / aa2;
    L[1][0] = (un * nx - vx) / ny;
    L[1][1] = (1.0 - nx * nx) / ny;
    L[1][2] = -nx;
    L[1][3] = 0;
  }
  ns[0] = a;
  ns[1] = vx;
  ns[2] = vy;
  ns[3] = ek;
  ns[4] = a * a / gm1 + ek;
}
template <int DIR>
__device__ __forceinline__ void ns2d_eigvecs(double g, const double u[4], double L[4][4], double R[4][4]) {
  double ns[5];
  ns2d_left<DIR>(g, u, L, ns);
  ns2d_right<DIR>(ns[0], ns[1], ns[2], ns[3], ns[4], R);
}

// rf-char selection for one characteristic field (Euler1DUpwindRF,
// Euler1DUpwind.c:160-173; NavierStokes2DUpwindRF, NavierStokes2DUpwind.c:152-166):
// upwind when the field's eigenvalue has one sign at the left, averaged and
// right states, else a local Lax-Friedrichs flux with the largest |eigenvalue|.
// With llf set, the local Lax-Friedrichs flux is taken for every field
// (Euler1DUpwindLLF, Euler1DUpwind.c:259-261; NavierStokes2DUpwindLLF,
// NavierStokes2DUpwind.c:248-250).
__device__ __forceinline__ double rf_pick(double eL, double eC, double eR, double ucL, double ucR, double fcL,
                                          double fcR, bool llf) {
  if (!llf && eL > 0 && eC > 0 && eR > 0) return fcL;
  if (!llf && eL < 0 && eC < 0 && eR < 0) return fcR;
  const double x1 = fabs(eL), x2 = fabs(eC), x3 = fabs(eR);
  const double mx1 = x1 > x2 ? x1 : x2, mx2 = x2 > x3 ? x2 : x3;
  const double alpha = mx1 > mx2 ? mx1 : mx2;
  return 0.5 * (fcL + fcR + alpha * (ucL - ucR));
}

// _NavierStokes2DGetFlowVar_, navierstokes2d.h:70-79
__device__ __forceinline__ void ns2d_flowvar(const double u[4], double gam, double &rho, double &vx, double &vy,
                                             double &e, double &P) {
  rho = u[0];
  vx = (rho == 0) ? 0 : u[1] / rho;
  vy = (rho == 0) ? 0 : u[2] / rho;
  e = u[3];
  const double vsq = (vx * vx) + (vy * vy);
  P = (e - 0.5 * rho * vsq) * (gam - 1.0);
}

// The flux along dir at one point (NavierStokes2DFlux.c:24-52 with
// navierstokes2d.h:70-110; Euler1DFlux.c:19 with euler1d.h:61-85): q(m) reads
// variable m of the point, put(m, value) writes component m of the flux.
template <class Q, class Put>
__device__ __forceinline__ void point_flux(int model, int dir, double gamma, int nv, Q q, Put put) {
  if (model == 1) {
    const double rho = q(0), v = q(1) / rho, e = q(2);
    const double P_ = (e - 0.5 * rho * v * v) * (gamma - 1.0);
    put(0, rho * v);
    put(1, rho * v * v + P_);
    put(2, (e + P_) * v);
    for (int m = 3; m < nv; m++) put(m, v * q(m));
  } else {
    const double rho = q(0);
    const double vx = (rho == 0) ? 0 : q(1) / rho;
    const double vy = (rho == 0) ? 0 : q(2) / rho;
    const double e = q(3);
    const double vsq = (vx * vx) + (vy * vy);
    const double P_ = (e - 0.5 * rho * vsq) * (gamma - 1.0);
    const double vn = dir == 0 ? vx : vy;
    put(0, rho * vn);
    if (dir == 0) {
      put(1, rho * vx * vx + P_);
      put(2, rho * vx * vy);
    } else {
      put(1, rho * vy * vx);
      put(2, rho * vy * vy + P_);
    }
    put(3, (e + P_) * vn);
    for (int m = 4; m < nv; m++) put(m, vn * q(m));
  }
}

// ---------------------------------------------------------------------------
// Upwinding at one interface.  uLc, uRc: the cells beside it; ud, fs:
// 0.5*(uR - uL) and 0.5*(fL + fR), the only combinations of the reconstructed
// values that the Roe and Rusanov fluxes use; fo: the flow part of the
// interface flux.
// ---------------------------------------------------------------------------
// Roe, NavierStokes2DUpwind.c:26-92: returns the species' dissipation
// coefficient.
template <int DIR>
__device__ __forceinline__ double roe_ns2d(double g, const double uLc[4], const double uRc[4], const double ud[4],
                                           const double fs[4], double fo[4]) {
  double ua[4], D[4], L[4][4], R[4][4];
  ns2d_roeavg(g, uLc, uRc, ua);
  ns2d_eigvals<DIR>(g, ua, D);
  ns2d_eigvecs<DIR>(g, ua, L, R);
  const double vn = D[3];
  const double delta = 0.000001, delta2 = delta * delta;
  const double Dsp = (fabs(vn) < delta ? (vn * vn + delta2) / (2 * delta) : fabs(vn));
#pragma unroll
  for (int m = 0; m < 4; m++) D[m] = (fabs(D[m]) < delta ? (D[m] * D[m] + delta2) / (2 * delta) : fabs(D[m]));
  // modA = R (D L), row-major sums in index order (matmult_native.h:21-34)
  double DL[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) DL[i][j] = D[i] * L[i][j];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    double us = 0.0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const double mA = R[i][0] * DL[0][j] + R[i][1] * DL[1][j] + R[i][2] * DL[2][j] + R[i][3] * DL[3][j];
      us += mA * ud[j];
    }
    fo[i] = fs[i] - us;
  }
  return Dsp;
}

// NavierStokes2DUpwindRusanov (NavierStokes2DUpwind.c:271-332): the largest of
// c + |v_n| at the two neighbouring cells and their Roe average.
template <int DIR>
__device__ __forceinline__ double rusanov_ns2d(double g, const double uLc[4], const double uRc[4]) {
  double ua[4];
  ns2d_roeavg(g, uLc, uRc, ua);
  auto speed = [&](const double u[4]) {
    double rho, vx, vy, e, P;
    ns2d_flowvar(u, g, rho, vx, vy, e, P);
    return sqrt(g * P / rho) + fabs(DIR == 0 ? vx : vy);
  };
  const double aL = speed(uLc), aR = speed(uRc), aA = speed(ua);
  const double m1 = aL > aR ? aL : aR, m2 = aR > aA ? aR : aA;  // max3, math_ops.h:30
  return m1 > m2 ? m1 : m2;
}

// NavierStokes2DUpwindRF (NavierStokes2DUpwind.c:106-187): L and R from the
// Roe average of the two reconstructed interface states uL, uR (not of the
// neighbouring cells); a field is upwinded by the signs of its eigenvalue at
// uL, uR and the average.  Species fields have eigenvalue vn, whose three
// values es returns, and identity eigenvectors.
template <int DIR>
__device__ __forceinline__ void rf_ns2d(double g, bool llf, const double uLk[4], const double uRk[4],
                                        const double fLk[4], const double fRk[4], double fo[4], double es[3]) {
  double ua[4], L[4][4], R[4][4], eL[4], eC[4], eR[4];
  ns2d_roeavg(g, uLk, uRk, ua);
  ns2d_eigvecs<DIR>(g, ua, L, R);
  ns2d_eigvals<DIR>(g, uLk, eL);
  ns2d_eigvals<DIR>(g, uRk, eR);
  ns2d_eigvals<DIR>(g, ua, eC);
  double fc[4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    // MatVecMult (matmult_native.h:119-130): row sums in index order
    const double ucL = L[m][0] * uLk[0] + L[m][1] * uLk[1] + L[m][2] * uLk[2] + L[m][3] * uLk[3];
    const double ucR = L[m][0] * uRk[0] + L[m][1] * uRk[1] + L[m][2] * uRk[2] + L[m][3] * uRk[3];
    const double fcL = L[m][0] * fLk[0] + L[m][1] * fLk[1] + L[m][2] * fLk[2] + L[m][3] * fLk[3];
    const double fcR = L[m][0] * fRk[0] + L[m][1] * fRk[1] + L[m][2] * fRk[2] + L[m][3] * fRk[3];
    fc[m] = rf_pick(eL[m], eC[m], eR[m], ucL, ucR, fcL, fcR, llf);
  }
#pragma unroll
  for (int i = 0; i < 4; i++) fo[i] = R[i][0] * fc[0] + R[i][1] * fc[1] + R[i][2] * fc[2] + R[i][3] * fc[3];
  es[0] = eL[3];
  es[1] = eC[3];
  es[2] = eR[3];
}

// Euler1DUpwindRoe (Euler1DUpwind.c:27-93): |A| = R |D| L of the average's
// eigenstructure, with the species' coefficient returned, and the flux from it
__device__ __forceinline__ double roe_matrix_e1d(const Eig3 &E, double A[3][3]) {
  double DL[3][3];
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++) DL[i][j] = fabs(E.D[i]) * E.L[i][j];
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++) A[i][j] = E.R[i][0] * DL[0][j] + E.R[i][1] * DL[1][j] + E.R[i][2] * DL[2][j];
  return fabs(E.D[0]);
}
__device__ __forceinline__ void roe_apply_e1d(const double A[3][3], const double ud[3], const double fs[3],
                                              double fo[3]) {
#pragma unroll
  for (int i = 0; i < 3; i++) {
    double us = 0.0;
#pragma unroll
    for (int j = 0; j < 3; j++) us += A[i][j] * ud[j];
    fo[i] = fs[i] - us;
  }
}
__device__ __forceinline__ double roe_e1d(double g, const double uLc[3], const double uRc[3], const double ud[3],
                                          const double fs[3], double fo[3]) {
  double a0, a1, a2, A[3][3];
  euler1d_roeavg(g, uLc[0], uLc[1], uLc[2], uRc[0], uRc[1], uRc[2], a0, a1, a2);
  Eig3 E;
  euler1d_eig(g, a0, a1, a2, E);
  const double c = roe_matrix_e1d(E, A);
  roe_apply_e1d(A, ud, fs, fo);
  return c;
}

// Euler1DUpwindRusanov (Euler1DUpwind.c:282-353); its wave speed is gamma P/rho
// + |u|, with no square root, as the reference computes it
__device__ __forceinline__ double rusanov_e1d(double g, const double uLc[3], const double uRc[3]) {
  double a0, a1, a2;
  euler1d_roeavg(g, uLc[0], uLc[1], uLc[2], uRc[0], uRc[1], uRc[2], a0, a1, a2);
  auto speed = [&](double rho, double mom, double e) {
    const double uvel = mom / rho, P = (e - 0.5 * rho * uvel * uvel) * (g - 1.0);
    return g * P / rho + fabs(uvel);
  };
  const double aL = speed(uLc[0], uLc[1], uLc[2]), aR = speed(uRc[0], uRc[1], uRc[2]);
  const double aA = speed(a0, a1, a2);
  const double m1 = aL > aR ? aL : aR, m2 = aR > aA ? aR : aA;  // max3, math_ops.h:30
  return m1 > m2 ? m1 : m2;
}

// rf-char (Euler1DUpwind.c:107-190) and llf-char (:199-266); es: the species'
// eigenvalue at the left cell, the average and the right cell
__device__ __forceinline__ void rf_e1d(double g, bool llf, const double uLc[3], const double uRc[3],
                                       const double uL[3], const double uR[3], const double fL[3],
                                       const double fR[3], double fo[3], double es[3]) {
  double a0, a1, a2;
  euler1d_roeavg(g, uLc[0], uLc[1], uLc[2], uRc[0], uRc[1], uRc[2], a0, a1, a2);
  Eig3 E, EL, ER;
  euler1d_eig(g, a0, a1, a2, E);
  // cell eigenvalues (euler1d.h:131-147) of the two neighbours
  euler1d_eig(g, uLc[0], uLc[1], uLc[2], EL);
  euler1d_eig(g, uRc[0], uRc[1], uRc[2], ER);
  double fc[3];
#pragma unroll
  for (int m = 0; m < 3; m++) {
    double ucL = 0, ucR = 0, fcL = 0, fcR = 0;
#pragma unroll
    for (int j = 0; j < 3; j++) {
      ucL += E.L[m][j] * uL[j];
      ucR += E.L[m][j] * uR[j];
      fcL += E.L[m][j] * fL[j];
      fcR += E.L[m][j] * fR[j];
    }
    fc[m] = rf_pick(EL.D[m], E.D[m], ER.D[m], ucL, ucR, fcL, fcR, llf);
  }
#pragma unroll
  for (int i = 0; i < 3; i++) fo[i] = E.R[i][0] * fc[0] + E.R[i][1] * fc[1] + E.R[i][2] * fc[2];
  // species rows: identity eigenvectors, eigenvalue v
  es[0] = EL.D[0];
  es[1] = E.D[0];
  es[2] = ER.D[0];
}

// Element at byte offset o of an array: the offset of a point is formed once for
// all planes, whose bases are the same for the block.
__device__ __forceinline__ const double &elem(const double *base, size_t o) {
  return *(const double *)((const char *)base + o);
}
__device__ __forceinline__ double &elem(double *base, size_t o) { return *(double *)((char *)base + o); }

// Block barrier that orders LDS accesses only: global loads and stores issued
// before it stay in flight (a __syncthreads also waits for those).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ---------------------------------------------------------------------------
// Ensemble indexing: block -> case, local work item
// ---------------------------------------------------------------------------
#define CASE_ARGS const CaseDev *__restrict__ cases, const int *__restrict__ blockcase, \
                  const int *__restrict__ firstblock, int stage
// Workgroups go to the eight XCDs in turn, each XCD with its own L2.  The tile
// kernels take their tiles in this order: each XCD gets one contiguous band of
// the case's nb tiles, so that the cache lines two neighbouring tiles share are
// fetched into one L2.  It is a bijection of 0..nb-1; a case whose blocks do not
// start on a multiple of eight keeps workgroup order.
__device__ __forceinline__ int xcd_order(int id, int nb, int first) {
  if (!PIAFS_XCD_ORDER || (first & 7)) return id;
  const int q = nb >> 3, r = nb & 7, x = id & 7, k = id >> 3;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + k;
}

// A plan of one case has no tables: a launch's first loads are then of the case
// itself, a memory round trip earlier.
#define CASE_PREAMBLE                                                      \
  const int cidx = blockcase ? blockcase[blockIdx.x] : 0;                  \
  const int first = blockcase ? firstblock[cidx] : 0;                      \
  const CaseDev &C = cases[cidx];                                          \
  const long t = (long)((int)blockIdx.x - first) * blockDim.x + threadIdx.x; \
  (void)stage;

}  // namespace

}  // namespace piafs
