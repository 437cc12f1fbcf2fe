// The hyperbolic interface flux of the schemes without line systems (WENO5 and
// upw5, component-wise or characteristic) in one pass over the stage state.
#include "viscous.hpp"

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

// The 64 interfaces of a block (item: this lane's, counted over the sweep).
template <int MODEL, int DIR, int KIND, bool CH>
__device__ __forceinline__ void weno_tile(const CaseDev &C, long item, int uw, Rows &sh) {
  constexpr int NF = MODEL == 1 ? 3 : 4;
  const SweepGeom &S = DIR ? C.Sy : C.Sx;
  const int nv = C.G.nv, N = S.N, nl = S.nlines, x = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const double g = C.P.gamma;
  const bool active = item < (long)(N + 1) * nl;
  const long it = active ? item : 0;
  const int l = (int)(it / (N + 1)), k = (int)(it % (N + 1));
  const long pl = S.plane, vs = (long)nl * (N + 1);
  const double *u = (DIR ? C.UT : C.U) + S.base + (long)l * S.line_stride + k;  // variable 0 right of the interface
  double *fI = (DIR ? C.fIy : C.fIx) + it;
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
      Eig3 E;
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
  const int mode = C.upwind;
  if (wave == uw) {
    double uLc[4], uRc[4], fo[4];
    if (MODEL == 1 || mode == 0 || mode == 3) cells(uLc, uRc);
    auto o = [&](int a, int m) { return sh.o[4 * a + m][x]; };
    if (mode == 0 || mode == 3) {
      double ud[4], fs[4], c;
#pragma unroll
      for (int m = 0; m < NF; m++) {
        ud[m] = 0.5 * (o(1, m) - o(0, m));
        fs[m] = 0.5 * (o(2, m) + o(3, m));
      }
      if (mode == 0) {
        if constexpr (MODEL == 1) c = roe_e1d(g, uLc, uRc, ud, fs, fo);
        else c = roe_ns2d<DIR>(g, uLc, uRc, ud, fs, fo);
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

// Reconstruction of the state and of its flux, and the upwinding, at every
// interface of both sweeps, from the stage state alone: cell fluxes are formed
// at the six stencil positions, so neither they nor the reconstructed values
// exist in memory.  The viscous fluxes, which need the stage state alone too,
// have the launch's first blocks.  Bound by FP64 issue on large grids and by the latency of
// the FP64 chains on small ones.  A block of four waves takes 64 interfaces, a
// wave a variable at a time: with a thread taking an interface through every
// variable the kernel needs 236 registers (characteristic 318), which leaves
// one or two waves per SIMD waiting on their own chains.  Per stage, cell
// fluxes, end interfaces, reconstruction and upwinding as separate passes ->
// one thread per interface -> this: 600 x 343, 11 variables, components 186 ->
// 146 -> 100 us; 500 x 100, 11 variables, characteristic 63 -> 48 -> 35;
// 201 x 201, 4 variables, characteristic 36 -> 28 -> 21; 1024-point line,
// characteristic 17 -> 8.2 -> 7.9.
__global__ void __launch_bounds__(256) k_weno(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage >= C.nstages) return;
  __shared__ union Lds {
    Rows rows;
    Prims prims;
  } lds;
  const int nvis = viscous_blocks(C);
  if ((int)(blockIdx.x - firstblock[cidx]) < nvis) {
    viscous_tile(C, (int)(blockIdx.x - firstblock[cidx]), lds.prims);
    return;
  }
  Rows &sh = lds.rows;
  const long nX = (long)(C.Sx.N + 1) * C.Sx.nlines;
  const int nbx = (int)((nX + 63) / 64);
  const int bid = (int)(blockIdx.x - firstblock[cidx]) - nvis;
  const int dir = bid < nbx ? 0 : 1;
  const long item = (long)(dir ? bid - nbx : bid) * 64 + (threadIdx.x & 63);
  const int uw = bid & 3;  // in turn, since a block's waves sit on the SIMDs in order
  const bool ch = C.R.characteristic != 0;
#define WENO(MODEL, DIR, KIND) \
  (ch ? weno_tile<MODEL, DIR, KIND, true>(C, item, uw, sh) : weno_tile<MODEL, DIR, KIND, false>(C, item, uw, sh))
#define WENO_ANY(KIND) (C.model == 1 ? WENO(1, 0, KIND) : dir ? WENO(2, 1, KIND) : WENO(2, 0, KIND))
  switch (C.R.kind) {
    case 1: WENO_ANY(1); break;
    case 2: WENO_ANY(2); break;
    case 3: WENO_ANY(3); break;
    case 4: WENO_ANY(4); break;
    default: WENO_ANY(0); break;
  }
#undef WENO_ANY
#undef WENO
}

// InterpolateInterfacesHyp of one array on the reference's layouts (a point's
// components contiguous).  Component-wise: one thread per (interface,
// variable) in memory order, so that its loads and its store are contiguous
// over a wave in either direction.  Characteristic: one thread per interface;
// L and R from the state u, species rows the identity.
template <int KIND>
__device__ __forceinline__ void dev_weno_at(const AosGrid &A, int model, double g, const ReconParams &R, int dir,
                                            bool left, const double *__restrict__ a, const double *__restrict__ u,
                                            long p, int v, double *__restrict__ fI) {
  const int nv = A.nv, N = dir ? A.ny : A.nx;
  const int k = (int)(dir ? p / A.nx : p % (N + 1)), l = (int)(dir ? p % A.nx : p / (N + 1));
  const long st = (dir ? A.nx + 2 * A.g : 1) * (long)nv;  // between positions of the line
  const long p0 = (A.ndims == 2 ? (long)((dir ? 0 : l) + A.g) * (A.nx + 2 * A.g) + ((dir ? l : 0) + A.g) : A.g) * nv;
  // position of stencil point q = 0 .. 4 (m3 .. p2)
  auto off = [&](int q) { return p0 + (left ? k - 3 + q : k + 2 - q) * st; };
  auto one = [&](int m) {
    return weno_value<KIND>(R, a[off(0) + m], a[off(1) + m], a[off(2) + m], a[off(3) + m], a[off(4) + m]);
  };
  double *out = fI + p * nv;
  if (!R.characteristic) {
    out[v] = one(v);
    return;
  }
  const double *cL = u + p0 + (k - 1) * st, *cR = u + p0 + k * st;
  int nf = 4;
  if (model == 1) {
    nf = 3;
    double a0, a1, a2, c[3];
    euler1d_roeavg(g, cL[0], cL[1], cL[2], cR[0], cR[1], cR[2], a0, a1, a2);
    Eig3 E;
    euler1d_eig(g, a0, a1, a2, E);
#pragma unroll
    for (int i = 0; i < 3; i++) {
      double s[5];
#pragma unroll
      for (int q = 0; q < 5; q++) {
        const double *x = a + off(q);
        s[q] = E.L[i][0] * x[0] + E.L[i][1] * x[1] + E.L[i][2] * x[2];
      }
      c[i] = weno_value<KIND>(R, s[0], s[1], s[2], s[3], s[4]);
    }
#pragma unroll
    for (int i = 0; i < 3; i++) out[i] = E.R[i][0] * c[0] + E.R[i][1] * c[1] + E.R[i][2] * c[2];
  } else {
    const double uLc[4] = {cL[0], cL[1], cL[2], cL[3]}, uRc[4] = {cR[0], cR[1], cR[2], cR[3]};
    double ua[4], L[4][4], Rm[4][4], c[4];
    ns2d_roeavg(g, uLc, uRc, ua);
    if (dir) ns2d_eigvecs<1>(g, ua, L, Rm);
    else ns2d_eigvecs<0>(g, ua, L, Rm);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      double s[5];
#pragma unroll
      for (int q = 0; q < 5; q++) {
        const double *x = a + off(q);
        s[q] = L[i][0] * x[0] + L[i][1] * x[1] + L[i][2] * x[2] + L[i][3] * x[3];
      }
      c[i] = weno_value<KIND>(R, s[0], s[1], s[2], s[3], s[4]);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = Rm[i][0] * c[0] + Rm[i][1] * c[1] + Rm[i][2] * c[2] + Rm[i][3] * c[3];
  }
  for (int m = nf; m < nv; m++) out[m] = one(m);
}

__global__ void __launch_bounds__(256) k_dev_weno(AosGrid A, int model, double g, ReconParams R, int dir, int left,
                                                  const double *__restrict__ a, const double *__restrict__ u,
                                                  double *__restrict__ fI) {
  const int N = dir ? A.ny : A.nx, nl = A.ndims == 2 ? (dir ? A.nx : A.ny) : 1;
  const int per = R.characteristic ? 1 : A.nv;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)(N + 1) * nl * per) return;
  const long p = t / per;
  const int v = (int)(t % per);
  switch (R.kind) {
    case 1: dev_weno_at<1>(A, model, g, R, dir, left != 0, a, u, p, v, fI); break;
    case 2: dev_weno_at<2>(A, model, g, R, dir, left != 0, a, u, p, v, fI); break;
    case 3: dev_weno_at<3>(A, model, g, R, dir, left != 0, a, u, p, v, fI); break;
    case 4: dev_weno_at<4>(A, model, g, R, dir, left != 0, a, u, p, v, fI); break;
    default: dev_weno_at<0>(A, model, g, R, dir, left != 0, a, u, p, v, fI); break;
  }
}

}  // namespace

void launch_dev_weno(const AosGrid &A, int model, double gamma, const ReconParams &R, int dir, bool left,
                     const double *a, const double *u, double *fI, hipStream_t s) {
  const long n = (long)((dir ? A.ny : A.nx) + 1) * (A.ndims == 2 ? (dir ? A.nx : A.ny) : 1) *
                 (R.characteristic ? 1 : A.nv);
  hipLaunchKernelGGL(k_dev_weno, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, A, model, gamma, R, dir,
                     left ? 1 : 0, a, u, fI);
}

KernFn weno_kernel() { return k_weno; }

}  // namespace piafs
