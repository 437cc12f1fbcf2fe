// The interface flux of the schemes without line systems, 64 interfaces a block.
// Include from .hip files only.
#pragma once

#include "device.hpp"

namespace piafs {

namespace {

// one interpolated value: Interp1PrimFifthOrderWENO.c:124-166 with the weights
// of weno_w, or upw5 (KIND 4)
template <int KIND>
__device__ __forceinline__ double weno_value(const ReconParams &R, double m3, double m2, double m1, double p1,
                                             double p2) {
  if (KIND == 4) return upw5_value(m3, m2, m1, p1, p2);
  double w1 = 0.1, w2 = 0.6, w3 = 0.3, f1, f2, f3;
  if (!R.no_limiting) weno_w<KIND>(0.1, 0.6, 0.3, m3, m2, m1, p1, p2, R.eps, w1, w2, w3);
  weno5_cands(m3, m2, m1, p1, p2, f1, f2, f3);
  return w1 * f1 + w2 * f2 + w3 * f3;
}

// left-biased (from positions k-3 .. k+1) and right-biased (k+2 .. k-2) value
// at interface k of the six values a[0..5] at k-3 .. k+2
template <int KIND>
__device__ __forceinline__ void weno_both(const ReconParams &R, const double a[6], double &vl, double &vr) {
  vl = weno_value<KIND>(R, a[0], a[1], a[2], a[3], a[4]);
  vr = weno_value<KIND>(R, a[5], a[4], a[3], a[2], a[1]);
}

// LDS of a block, rows of 64 doubles, one per interface of its tile
constexpr int kHeld = 7;  // species a block reconstructs at a time (a layer's)
struct Rows {
  double fl[24][64];  // flow flux at the six stencil positions, [4 * position + variable]
  double left[16][64];  // left eigenvectors, by rows
  double vn[6][64];   // velocity along the sweep at the six positions
  double o[16][64];   // uL, uR, fL, fR of the flow variables, [4 * array + variable]
  double eig[9][64];  // what the right eigenvectors need
  double es[3][64];   // the species' dissipation coefficient, or their eigenvalue at left, average, right
  // the species' uL, uR, fL, fR, [4 * species + array], once fl and left are done with
  __device__ __forceinline__ double *held(int r) { return fl[0] + 64 * r; }
};
static_assert(4 * kHeld <= 24 + 16, "held rows lie in fl and left");

// The 64 interfaces of a 256-thread block, a lane each.  u: variable 0 at the
// position right of the lane's interface, planes pl apart; fI: where the flux of
// variable 0 goes, variables vs apart, if active.
template <int MODEL, int DIR, int KIND, bool CH>
__device__ __forceinline__ void weno_tile(const CaseDev &C, const double *__restrict__ u, long pl, double *fI, long vs,
                                          bool active, int uw, Rows &sh) {
  constexpr int NF = MODEL == 1 ? 3 : 4;
  const int nv = C.G.nv, x = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const double g = C.P.gamma;
  const int mode = C.upwind;
  // Roe in 1D: the last wave has no variable to reconstruct, so it forms |A| of
  // the two cells' average then and upwinds
  const bool early = MODEL == 1 && mode == 0;
  if (early) uw = 3;
  Eig3 E;
  double A[3][3], es1 = 0.0;
  auto cells = [&](double uLc[4], double uRc[4]) {  // the two cells beside the interface
#pragma unroll
    for (int m = 0; m < NF; m++) {
      uLc[m] = u[m * pl - 1];
      uRc[m] = u[m * pl];
    }
  };
  // 1. the flow's flux and velocity at the six positions, shared out over the
  // waves; characteristic: the last wave takes the eigenvectors of the Roe
  // average of the two cells instead (WENOFifthOrderCalculateWeights.c:761-930)
  if (!CH || wave < 3) {
    for (int p = wave; p < 6; p += CH ? 3 : 4) {
      double q[4];
#pragma unroll
      for (int m = 0; m < NF; m++) q[m] = u[m * pl + p - 3];
      point_flux(MODEL, DIR, g, NF, [&](int m) { return q[m]; }, [&](int m, double f) { sh.fl[4 * p + m][x] = f; });
      if (nv > NF) sh.vn[p][x] = MODEL == 2 && q[0] == 0 ? 0 : q[1 + DIR] / q[0];
    }
  } else {
    double uLc[4], uRc[4];
    cells(uLc, uRc);
    if constexpr (MODEL == 1) {
      double a0, a1, a2;
      euler1d_roeavg(g, uLc[0], uLc[1], uLc[2], uRc[0], uRc[1], uRc[2], a0, a1, a2);
      euler1d_eig(g, a0, a1, a2, E);
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
          sh.left[4 * i + j][x] = E.L[i][j];
          sh.eig[3 * i + j][x] = E.R[i][j];
        }
    } else {
      double ua[4], L[4][4], ns[5];
      ns2d_roeavg(g, uLc, uRc, ua);
      ns2d_left<DIR>(g, ua, L, ns);
#pragma unroll
      for (int i = 0; i < 16; i++) sh.left[i][x] = L[i >> 2][i & 3];
#pragma unroll
      for (int i = 0; i < 5; i++) sh.eig[i][x] = ns[i];
    }
  }
  lds_barrier();
  // 2. wave v: flow variable (or characteristic field) v of the state and of
  // the flux, products summed in index order as MatVecMult does
  if (wave < NF) {
    const int v = wave;
    double a[6], vl, vr;
#pragma unroll
    for (int src = 0; src < 2; src++) {
#pragma unroll
      for (int p = 0; p < 6; p++) {
        auto q = [&](int m) { return src ? sh.fl[4 * p + m][x] : u[m * pl + p - 3]; };
        if (CH) {
          double y = sh.left[4 * v][x] * q(0);
#pragma unroll
          for (int m = 1; m < NF; m++) y = y + sh.left[4 * v + m][x] * q(m);
          a[p] = y;
        } else {
          a[p] = q(v);
        }
      }
      weno_both<KIND>(C.R, a, vl, vr);
      sh.o[4 * (2 * src) + v][x] = vl;
      sh.o[4 * (2 * src + 1) + v][x] = vr;
    }
  } else if (early) {
    if constexpr (MODEL == 1) {
      if (!CH) {
        double uLc[4], uRc[4], a0, a1, a2;
        cells(uLc, uRc);
        euler1d_roeavg(g, uLc[0], uLc[1], uLc[2], uRc[0], uRc[1], uRc[2], a0, a1, a2);
        euler1d_eig(g, a0, a1, a2, E);
      }
      es1 = roe_matrix_e1d(E, A);
    }
  }
  lds_barrier();
  // 3. characteristic: back to the flow variables, wave s array s of uL, uR, fL, fR
  // (Interp1PrimFifthOrderWENOChar.c:89-201)
  if (CH) {
    double c[4];
#pragma unroll
    for (int m = 0; m < NF; m++) c[m] = sh.o[4 * wave + m][x];
    if constexpr (MODEL == 1) {
#pragma unroll
      for (int i = 0; i < 3; i++)
        sh.o[4 * wave + i][x] = sh.eig[3 * i][x] * c[0] + sh.eig[3 * i + 1][x] * c[1] + sh.eig[3 * i + 2][x] * c[2];
    } else {
      double R[4][4];
      ns2d_right<DIR>(sh.eig[0][x], sh.eig[1][x], sh.eig[2][x], sh.eig[3][x], sh.eig[4][x], R);
#pragma unroll
      for (int i = 0; i < 4; i++)
        sh.o[4 * wave + i][x] = R[i][0] * c[0] + R[i][1] * c[1] + R[i][2] * c[2] + R[i][3] * c[3];
    }
    lds_barrier();
  }
  // 4. wave uw: the flow's interface flux, while the other waves begin the species
  if (wave == uw) {
    double uLc[4], uRc[4], fo[4];
    if (!early && (MODEL == 1 || mode == 0 || mode == 3)) cells(uLc, uRc);
    auto o = [&](int a, int m) { return sh.o[4 * a + m][x]; };
    if (mode == 0 || mode == 3) {
      double ud[4], fs[4], c;
#pragma unroll
      for (int m = 0; m < NF; m++) {
        ud[m] = 0.5 * (o(1, m) - o(0, m));
        fs[m] = 0.5 * (o(2, m) + o(3, m));
      }
      if (mode == 0) {
        if constexpr (MODEL == 1) {
          roe_apply_e1d(A, ud, fs, fo);
          c = es1;
        } else c = roe_ns2d<DIR>(g, uLc, uRc, ud, fs, fo);
      } else {
        if constexpr (MODEL == 1) c = rusanov_e1d(g, uLc, uRc);
        else c = rusanov_ns2d<DIR>(g, uLc, uRc);
#pragma unroll
        for (int m = 0; m < NF; m++) fo[m] = fs[m] - c * ud[m];
      }
      if (nv > NF) sh.es[0][x] = c;
    } else {
      double b[4][4], e[3];
#pragma unroll
      for (int i = 0; i < 16; i++)
        if ((i & 3) < NF) b[i >> 2][i & 3] = o(i >> 2, i & 3);
      if constexpr (MODEL == 1) rf_e1d(g, mode == 2, uLc, uRc, b[0], b[1], b[2], b[3], fo, e);
      else rf_ns2d<DIR>(g, mode == 2, b[0], b[1], b[2], b[3], fo, e);
      if (nv > NF)
#pragma unroll
        for (int m = 0; m < 3; m++) sh.es[m][x] = e[m];
    }
    if (active)
#pragma unroll
      for (int m = 0; m < NF; m++) fI[m * vs] = fo[m];
  }
  // 5. the species, kHeld at a time, dealt out from the wave after uw
  // (identity eigenvectors: component-wise in every scheme)
  const int first = (wave - uw + 3) & 3;
  for (int m0 = NF; m0 < nv; m0 += kHeld) {
    const int n = min(kHeld, nv - m0);
    for (int h = first; h < n; h += 4) {
      double a[6], vl, vr;
#pragma unroll
      for (int p = 0; p < 6; p++) a[p] = u[(m0 + h) * pl + p - 3];
      weno_both<KIND>(C.R, a, vl, vr);
      sh.held(4 * h)[x] = vl;
      sh.held(4 * h + 1)[x] = vr;
#pragma unroll
      for (int p = 0; p < 6; p++) a[p] = sh.vn[p][x] * a[p];
      weno_both<KIND>(C.R, a, vl, vr);
      sh.held(4 * h + 2)[x] = vl;
      sh.held(4 * h + 3)[x] = vr;
    }
    if (m0 == NF) lds_barrier();  // es is written; each wave reads back its own species only
    for (int h = first; h < n; h += 4) {
      const double uL = sh.held(4 * h)[x], uR = sh.held(4 * h + 1)[x];
      const double fL = sh.held(4 * h + 2)[x], fR = sh.held(4 * h + 3)[x];
      const double f = mode == 0 || mode == 3 ? 0.5 * (fL + fR) - sh.es[0][x] * (0.5 * (uR - uL))
                                              : rf_pick(sh.es[0][x], sh.es[1][x], sh.es[2][x], uL, uR, fL, fR, mode == 2);
      if (active) fI[(m0 + h) * vs] = f;
    }
  }
}

}  // namespace

}  // namespace piafs
