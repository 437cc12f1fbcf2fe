// The viscous fluxes of navierstokes2d.  Include from .hip files only.
#pragma once

#include "device.hpp"

namespace piafs {

namespace {

// ---------------------------------------------------------------------------
// Parabolic term (navierstokes2d): NavierStokes2DParabolicFunction.c:41-204.
// Serial-run semantics: d/dx of Q is evaluated on interior rows only and d/dy
// on interior columns only (FirstDerivativeFourthOrder.c:66-71 loops over the
// interior lines of the other dimension); elsewhere the derivative is zero.
// ---------------------------------------------------------------------------
struct Prim {
  double vx, vy, T;
};
__device__ __forceinline__ Prim prim_of(double gam, double rho, double mx, double my, double e) {
  const double vx = (rho == 0) ? 0 : mx / rho, vy = (rho == 0) ? 0 : my / rho;
  const double vsq = (vx * vx) + (vy * vy);
  const double P = (e - 0.5 * rho * vsq) * (gam - 1.0);
  Prim r;
  r.vx = vx;
  r.vy = vy;
  r.T = gam * P / rho;
  return r;
}
__device__ __forceinline__ Prim prim_at(long plane, double gam, const double *U, long p) {
  return prim_of(gam, U[p], U[plane + p], U[2 * plane + p], U[3 * plane + p]);
}

// FirstDerivativeFourthOrder.c:39-132 (par4) / FirstDerivativeFirstOrder.c (bias +1)
// of the three primitives at position i of a line of N interior points, P(k)
// the primitives at position k (component c: P(k, c)).
template <class F>
__device__ __forceinline__ void deriv_prim(int g, bool par4, int i, int N, F P, double out[3]) {
#pragma unroll
  for (int c = 0; c < 3; c++) {
    if (par4) {
      const double t12 = 1.0 / 12.0;
      if (i == -g)
        out[c] = (-25 * P(i, c) + 48 * P(i + 1, c) - 36 * P(i + 2, c) + 16 * P(i + 3, c) - 3 * P(i + 4, c)) * t12;
      else if (i == -g + 1)
        out[c] = (-3 * P(i - 1, c) - 10 * P(i, c) + 18 * P(i + 1, c) - 6 * P(i + 2, c) + P(i + 3, c)) * t12;
      else if (i == N + g - 2)
        out[c] = (-P(i - 3, c) + 6 * P(i - 2, c) - 18 * P(i - 1, c) + 10 * P(i, c) + 3 * P(i + 1, c)) * t12;
      else if (i == N + g - 1)
        out[c] = (3 * P(i - 4, c) - 16 * P(i - 3, c) + 36 * P(i - 2, c) - 48 * P(i - 1, c) + 25 * P(i, c)) * t12;
      else
        out[c] = (P(i - 2, c) - 8 * P(i - 1, c) + 8 * P(i + 1, c) - P(i + 2, c)) * t12;
    } else if (i == -g) {
      out[c] = P(i + 1, c) - P(i, c);
    } else if (i == N + g - 1) {
      out[c] = P(i, c) - P(i - 1, c);
    } else {
      out[c] = 1.0 * P(i + 1, c) - 1.0 * P(i, c) + 0.0 * P(i - 1, c);
    }
  }
}

// Viscous fluxes (NavierStokes2DParabolicFunction.c:112-143 and :155-186),
// Sutherland viscosity and the conductivity law of navierstokes2d.h:315-331
// (raiseto(x,1.5) = exp(1.5 log x), include/math_ops.h:40), from the derivatives
// of velocity and temperature, each scaled by dxinv
// (NavierStokes2DParabolicFunction.c:96-106).  With the derivative exchange
// along a periodic dimension (xchg, MPIExchangeBoundariesnD.c:109-167 as called
// at NavierStokes2DParabolicFunction.c:91-94), a ghost point of an interior
// line across that dimension takes the unscaled derivatives of its periodic
// image, scaled by its own dxinv; corners are not exchanged, and never read.
// FV planes: 0..2 = x-flux components 1..3, 3..5 = y-flux components 1..3.
//
// A 32 x 8 tile of ghosted points per block, among the blocks of the launch
// that also reads the stage state only (k_flux, or k_weno), so that neither
// waits for the other.  Bound by latency on small grids
// and by HBM on large ones: the primitives of the tile and of the four points
// beside it (one-sided stencils reach that far) are formed once into LDS, 2.25
// division chains a thread instead of 21 in two passes with the derivatives
// in memory between them.  A block's chain took 17000 cycles with the points
// formed one after the other and a branch per kind of stencil, now 7500 (cavity
// 128 x 128, k_weno's launch 9.3 -> 7.9 us).
constexpr int kVisX = 32, kVisY = 8, kVisH = 4;
__host__ __device__ inline int viscous_blocks(const CaseDev &C) {
  if (C.G.ndims != 2 || !C.P.viscous) return 0;
  return ((C.G.nxg + kVisX - 1) / kVisX) * ((C.G.nyg + kVisY - 1) / kVisY);
}
// FirstDerivativeFourthOrder.c's stencil at position i as deriv_prim has it, for
// a wave whose lanes have different ones: five coefficients in the order of the
// sum, from position i + off on (the middle one is zero, and its term left out,
// away from the ends)
struct Stencil5 {
  int off;
  double c[5];
};
__device__ __forceinline__ Stencil5 stencil5(int g, int i, int N) {
  Stencil5 s = {-2, {1.0, -8.0, 0.0, 8.0, -1.0}};
  if (i == -g) s = {0, {-25.0, 48.0, -36.0, 16.0, -3.0}};
  if (i == -g + 1) s = {-1, {-3.0, -10.0, 18.0, -6.0, 1.0}};
  if (i == N + g - 2) s = {-3, {-1.0, 6.0, -18.0, 10.0, 3.0}};
  if (i == N + g - 1) s = {-4, {3.0, -16.0, 36.0, -48.0, 25.0}};
  return s;
}
// p: the value at position i, st apart
__device__ __forceinline__ double derive5(const Stencil5 &s, const double *p, int st) {
  const double t12 = 1.0 / 12.0, *q = p + s.off * st;
  double x = s.c[0] * q[0] + s.c[1] * q[st];
  const double y = x + s.c[2] * q[2 * st];
  x = s.c[2] == 0.0 ? x : y;
  x = x + s.c[3] * q[3 * st];
  x = x + s.c[4] * q[4 * st];
  return x * t12;
}

struct Prims {
  double pr[3][kVisY + 2 * kVisH][kVisX + 2 * kVisH];
};
// tile b of a 256-thread block
__device__ __forceinline__ void viscous_tile(const CaseDev &C, int b, Prims &sh) {
  const Grid &G = C.G;
  const PhysParams &P = C.P;
  auto &pr = sh.pr;
  const int tiles = (G.nxg + kVisX - 1) / kVisX;
  const int I0 = (b % tiles) * kVisX, J0 = (b / tiles) * kVisY;  // ghosted indices
  const double gam = P.gamma;
  const int tx = threadIdx.x & (kVisX - 1), ty = threadIdx.x / kVisX;
  // a thread forms its own point's primitives, those of one of the four rows below
  // and above, and the first 64 threads those of a point in the columns beside;
  // outside the grid the nearest point's, which no stencil reads, so that all loads
  // go out before the first is needed
  const int side = threadIdx.x & (2 * kVisH - 1);
  const int row[3] = {ty + kVisH, ty < kVisH ? ty : ty + kVisY, (int)threadIdx.x / (2 * kVisH) + kVisH};
  const int col[3] = {tx + kVisH, tx + kVisH, side < kVisH ? side : side + kVisX};
  const int nfill = threadIdx.x < 2 * kVisH * kVisY ? 3 : 2;
  double q[3][4];
#pragma unroll
  for (int f = 0; f < 3; f++)
    if (f < nfill) {
      const int I = min(max(I0 + col[f] - kVisH, 0), G.nxg - 1), J = min(max(J0 + row[f] - kVisH, 0), G.nyg - 1);
#pragma unroll
      for (int m = 0; m < 4; m++) q[f][m] = elem(C.U + m * G.plane, 8 * ((size_t)J * G.nxg + I));
    }
#pragma unroll
  for (int f = 0; f < 3; f++)
    if (f < nfill) {
      const Prim w = prim_of(gam, q[f][0], q[f][1], q[f][2], q[f][3]);
      pr[0][row[f]][col[f]] = w.vx;
      pr[1][row[f]][col[f]] = w.vy;
      pr[2][row[f]][col[f]] = w.T;
    }
  lds_barrier();
  const int I = I0 + tx, J = J0 + ty;
  if (I >= G.nxg || J >= G.nyg) return;
  const int i = I - G.g, j = J - G.g;
  const bool iin = i >= 0 && i < G.nx, jin = j >= 0 && j < G.ny;
  if (!iin && !jin) return;  // corners are never read
  double dx[3] = {0, 0, 0}, dy[3] = {0, 0, 0};
  // derivatives along x on interior rows, along y on interior columns
  const bool ex = P.xchg[0] && jin && !iin, ey = P.xchg[1] && iin && !jin;
  auto far = [&](int x, int y, int c) {  // a point outside the tile's reach
    const Prim q = prim_at(G.plane, gam, C.U, (long)(y + G.g) * G.nxg + (x + G.g));
    return c == 0 ? q.vx : c == 1 ? q.vy : q.T;
  };
  if (ex) {  // both derivatives of the image in x
    const int si = i < 0 ? i + G.nx : i - G.nx;
    deriv_prim(G.g, P.par4, si, G.nx, [&](int k, int c) { return far(k, j, c); }, dx);
    deriv_prim(G.g, P.par4, j, G.ny, [&](int k, int c) { return far(si, k, c); }, dy);
  } else if (ey) {
    const int sj = j < 0 ? j + G.ny : j - G.ny;
    deriv_prim(G.g, P.par4, i, G.nx, [&](int k, int c) { return far(k, sj, c); }, dx);
    deriv_prim(G.g, P.par4, sj, G.ny, [&](int k, int c) { return far(i, k, c); }, dy);
  } else if (P.par4) {
    const Stencil5 sx = stencil5(G.g, i, G.nx), sy = stencil5(G.g, j, G.ny);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const double *p = &pr[c][ty + kVisH][tx + kVisH];
      const double x = derive5(sx, p, 1), y = derive5(sy, p, kVisX + 2 * kVisH);
      dx[c] = jin ? x : 0.0;
      dy[c] = iin ? y : 0.0;
    }
  } else {
    if (jin)
      deriv_prim(G.g, P.par4, i, G.nx, [&](int k, int c) { return pr[c][ty + kVisH][tx + kVisH + k - i]; }, dx);
    if (iin)
      deriv_prim(G.g, P.par4, j, G.ny, [&](int k, int c) { return pr[c][ty + kVisH + k - j][tx + kVisH]; }, dy);
  }
  const double sx = C.dxinv[G.g + i], sy = C.dxinv[(G.nx + 2 * G.g) + G.g + j];
  const double ux = dx[0] * sx, vx = dx[1] * sx, Tx = dx[2] * sx;
  const double uy = dy[0] * sy, vy = dy[1] * sy, Ty = dy[2] * sy;
  const double qx = pr[0][ty + kVisH][tx + kVisH], qy = pr[1][ty + kVisH][tx + kVisH];
  const double Td = pr[2][ty + kVisH][tx + kVisH] * P.Tref;
  const double r15 = exp(1.5 * log(Td / P.T0));
  const double mu = r15 * (P.T0 + P.TS) / (Td + P.TS);
  const double kap = r15 * P.kappa_num / (Td + P.TA * exp(-P.TB / Td));
  const double muRe = mu * P.inv_Re;
  const double kc = kap * P.inv_Re * P.inv_gm1 * P.inv_Pr;
  const long pl = (long)G.nxg * G.nyg, p = (long)J * G.nxg + I;
  double *FV = C.FV;
  const double txx = P.two_third * muRe * (2 * ux - vy);
  const double txy = muRe * (uy + vx);
  FV[p] = txx;
  FV[pl + p] = txy;
  FV[2 * pl + p] = qx * txx + qy * txy + kc * Tx;
  const double tyx = muRe * (uy + vx);
  const double tyy = P.two_third * muRe * (-ux + 2 * vy);
  FV[3 * pl + p] = tyx;
  FV[4 * pl + p] = tyy;
  FV[5 * pl + p] = qx * tyx + qy * tyy + kc * Ty;
}

}  // namespace

}  // namespace piafs
