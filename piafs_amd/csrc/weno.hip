// The hyperbolic interface flux of the schemes without line systems (WENO5 and
// upw5, component-wise or characteristic) in one pass over the stage state.
#include "viscous.hpp"
#include "weno.hpp"

namespace piafs {

namespace {

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
// 146 -> 95 us; 500 x 100, 11 variables, characteristic 63 -> 48 -> 35;
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
  if ((int)blockIdx.x - first < nvis) {
    viscous_tile(C, (int)blockIdx.x - first, lds.prims);
    return;
  }
  Rows &sh = lds.rows;
  const long nX = (long)(C.Sx.N + 1) * C.Sx.nlines;
  const int nbx = (int)((nX + 63) / 64);
  const int bid = (int)blockIdx.x - first - nvis;
  const int dir = bid < nbx ? 0 : 1;
  const long item = (long)(dir ? bid - nbx : bid) * 64 + (threadIdx.x & 63);
  const int uw = bid & 3;  // in turn, since a block's waves sit on the SIMDs in order
  const bool ch = C.R.characteristic != 0;
  const SweepGeom &S = dir ? C.Sy : C.Sx;
  const long vs = (long)S.nlines * (S.N + 1);
  const bool active = item < vs;
  const long it = active ? item : 0;
  const double *u = (dir ? C.UT : C.U) + S.base + (it / (S.N + 1)) * S.line_stride + it % (S.N + 1);
  double *fI = (dir ? C.fIy : C.fIx) + it;
#define WENO(MODEL, DIR, KIND)                                                             \
  (ch ? weno_tile<MODEL, DIR, KIND, true>(C, u, S.plane, fI, vs, active, uw, sh) \
      : weno_tile<MODEL, DIR, KIND, false>(C, u, S.plane, fI, vs, active, uw, sh))
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
