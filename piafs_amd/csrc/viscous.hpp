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
__device__ __forceinline__ Prim prim_at(long plane, double gam, const double *U, long p) {
  const double rho = U[p];
  const double vx = (rho == 0) ? 0 : U[plane + p] / rho, vy = (rho == 0) ? 0 : U[2 * plane + p] / rho;
  const double e = U[3 * plane + p];
  const double vsq = (vx * vx) + (vy * vy);
  const double P = (e - 0.5 * rho * vsq) * (gam - 1.0);
  Prim r;
  r.vx = vx;
  r.vy = vy;
  r.T = gam * P / rho;
  return r;
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
// divisions chains a thread instead of 21 in two passes with the derivatives
// in memory between them.
constexpr int kVisX = 32, kVisY = 8, kVisH = 4;
__host__ __device__ inline int viscous_blocks(const CaseDev &C) {
  if (C.G.ndims != 2 || !C.P.viscous) return 0;
  return ((C.G.nxg + kVisX - 1) / kVisX) * ((C.G.nyg + kVisY - 1) / kVisY);
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
  auto fill = [&](int a, int c) {  // LDS position (row a, column c)
    const int I = I0 + c - kVisH, J = J0 + a - kVisH;
    if (I < 0 || I >= G.nxg || J < 0 || J >= G.nyg) return;
    const Prim q = prim_at(G.plane, gam, C.U, (long)J * G.nxg + I);
    pr[0][a][c] = q.vx;
    pr[1][a][c] = q.vy;
    pr[2][a][c] = q.T;
  };
  const int tx = threadIdx.x & (kVisX - 1), ty = threadIdx.x / kVisX;
  fill(ty + kVisH, tx + kVisH);
  // four rows below and four above, then the columns beside the tile
  fill(ty < kVisH ? ty : ty + kVisY, tx + kVisH);
  if (threadIdx.x < 2 * kVisH * kVisY) {
    const int c = threadIdx.x & (2 * kVisH - 1), r = threadIdx.x / (2 * kVisH);
    fill(r + kVisH, c < kVisH ? c : c + kVisX);
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
