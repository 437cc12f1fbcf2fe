// HIP kernels for gfx950 (MI355X): the PIAFS hyperbolic/parabolic/source
// right-hand side and the explicit Runge-Kutta stage algebra, FP64 throughout.
//
// Arithmetic follows the reference's association order term by term (the
// file:line of the formula being restated is given at each device function),
// and the library is compiled without floating-point contraction so that the
// rounding of every +, -, *, / and sqrt matches the reference build.
#include "device.hpp"
#include "boundary.hpp"
#include "teams.hpp"
#include "viscous.hpp"

#include <cstdio>
#include <cstring>
#include <type_traits>

namespace piafs {

namespace {

constexpr int TB = 256;  // threads per block

inline unsigned nblk(long n, int tb = TB) { return (unsigned)((n + tb - 1) / tb); }

// ---------------------------------------------------------------------------
// Stage state + boundary conditions.
// TimeRK.c:46-57 (U = u + sum_j dt*A[s][j]*Udot_j, zero coefficients skipped:
// adding 0*Udot leaves U unchanged), then ApplyBoundaryConditions
// (BCPeriodic.c:22-62: ghost <- opposite interior; BCExtrapolate.c:16-51:
// mirror copy).  Each ghost point is evaluated at its boundary source point,
// which equals applying the BC to the stage state.  Points outside every
// boundary zone (the corners) are zero, as in the reference where they are
// never written.
// ---------------------------------------------------------------------------
// `stage` arguments with this bit leave the fused cases out
constexpr int kUnfused = 1 << 8;
__device__ __forceinline__ bool skipped(const CaseDev &C, int stage) { return (stage & kUnfused) && C.fused; }

__device__ __forceinline__ double stage_value(const CaseDev &C, int s, long p) {
  double val = C.u[p];
  const int ns = C.nstages;
  for (int j = 0; j < s; j++) {
    const double a = C.dt * C.A[s * ns + j];
    if (a != 0.0) val += a * C.Udot[j][p];
  }
  return val;
}

// Ghost points of the stage state, one thread per (variable, ghost point):
// the g rows below and above the interior (full ghosted width), then the g
// columns left and right of it (interior height).  Written to both layouts.

__host__ __device__ inline long ghost_points(const Grid &G) {
  return G.ndims == 1 ? 2L * G.g : 2L * G.gy * G.nxg + 2L * G.g * G.ny;
}

// state(p): the state at offset p; U: where the ghost points go, in the natural layout
template <class V>
__device__ __forceinline__ void ghost_body(const CaseDev &C, long t, V state, double *U) {
  const Grid &G = C.G;
  const long ng = ghost_points(G);
  if (t >= ng * G.nv) return;
  const int v = (int)(t / ng);
  long q = t % ng;
  int i, j = 0;
  if (G.ndims == 1) {
    i = (q < G.g) ? (int)q - G.g : G.nx + (int)(q - G.g);
  } else if (q < 2L * G.gy * G.nxg) {
    const int row = (int)(q / G.nxg);
    i = (int)(q % G.nxg) - G.g;
    j = row < G.gy ? row - G.gy : G.ny + (row - G.gy);
  } else {
    q -= 2L * G.gy * G.nxg;
    const int col = (int)(q / G.ny);
    j = (int)(q % G.ny);
    i = col < G.g ? col - G.g : G.nx + (col - G.g);
  }
  const double val = ghost_value(C, v, i, j, [&](int m, int a, int b) {
    return state((long)m * G.plane + (long)(b + G.gy) * G.nxg + (a + G.g));
  });
  const long pl = (long)v * G.plane;
  U[pl + (long)(j + G.gy) * G.nxg + (i + G.g)] = val;
  if (G.ndims == 2) C.UT[pl + (long)(i + G.g) * G.nyg + (j + G.gy)] = val;
}

// blocks of the interior points, padded to a multiple of eight for xcd_order;
// the blocks of the ghost points follow (they read the solution, not the stage
// state, so neither waits for the other)
__host__ __device__ inline int stage_blocks(const Grid &G, int st) {
  const long n = G.ndims == 1 ? ((long)G.nx * G.nv + TB - 1) / TB
                              : (long)((G.nx + st - 1) / st) * ((G.ny + st - 1) / st) * G.nv;
  return (int)((n + 7) & ~7L);
}

template <int ST>
__device__ __forceinline__ void stage_body(CASE_ARGS) {
  CASE_PREAMBLE
  const int s = stage & 0xFF;
  if (s >= C.nstages || skipped(C, stage)) return;
  const Grid &G = C.G;
  const int bid = (int)blockIdx.x - first, ns = stage_blocks(G, ST);
  if (bid >= ns) {
    ghost_body(C, t - (long)ns * TB, [&](long p) { return stage_value(C, s, p); }, C.U);
    return;
  }
  if (G.ndims == 1) {
    if (t >= (long)G.nx * G.nv) return;
    const int v = (int)(t / G.nx), i = (int)(t % G.nx);
    const long p = (long)v * G.plane + i + G.g;
    C.U[p] = stage_value(C, s, p);
    return;
  }
  // 2D interior: ST x ST tiles, 256 threads; natural write, then transposed
  // write via LDS.
  constexpr int SR = 256 / ST;
  __shared__ double tile[ST][ST + 1];
  const int ntx = (G.nx + ST - 1) / ST, nty = (G.ny + ST - 1) / ST;
  // (64-point tiles: workgroup order, which timed faster for them at 4096^2);
  // the case's block count is padded to a multiple of eight
  const int nb = G.nv * ntx * nty;
  const int id = ST == 32 ? xcd_order(bid, ns, first) : bid;
  if (id >= nb) return;
  const int v = id / (ntx * nty), rem = id % (ntx * nty);
  const int i0 = (rem % ntx) * ST, j0 = (rem / ntx) * ST;
  const int tx = threadIdx.x & (ST - 1), ty = threadIdx.x / ST;
  const long pl = (long)v * G.plane;
  for (int r = ty; r < ST; r += SR) {
    const int i = i0 + tx, j = j0 + r;
    double val = 0.0;
    if (i < G.nx && j < G.ny) {
      const long p = pl + (long)(j + G.gy) * G.nxg + (i + G.g);
      val = stage_value(C, s, p);
      C.U[p] = val;
    }
    tile[r][tx] = val;
  }
  __syncthreads();
  for (int r = ty; r < ST; r += SR) {
    const int i = i0 + r, j = j0 + tx;
    if (i < G.nx && j < G.ny) C.UT[pl + (long)(i + G.g) * G.nyg + (j + G.gy)] = tile[tx][r];
  }
}

// 32 x 32 tiles, or 64 x 64 when every case of the plan has at least
// 2048 x 2048 points (rows of 512 B in both layouts; 16 % faster there, 12 %
// slower at 1024 x 1024, where the smaller tiles give twice the blocks)
__global__ void __launch_bounds__(256) k_stage(CASE_ARGS) { stage_body<32>(cases, blockcase, firstblock, stage); }
__global__ void __launch_bounds__(256) k_stage64(CASE_ARGS) { stage_body<64>(cases, blockcase, firstblock, stage); }

// the ghost points alone, for the boundary-fill operator
__global__ void __launch_bounds__(256) k_ghost(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage < C.nstages) ghost_body(C, t, [&](long p) { return stage_value(C, stage, p); }, C.U);
}
// those of the state k_next wrote, of the cases with faces it does not fill
__global__ void __launch_bounds__(256) k_ghost_next(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage < C.nstages) ghost_body(C, t, [&](long p) { return C.Un[p]; }, C.Un);
}

// ---------------------------------------------------------------------------
// Cell-centred flux at every position of every interior line, both sweeps:
// the x-sweep from the natural state, the y-sweep from the transposed copy.
// NavierStokes2DFlux.c:24-52 (navierstokes2d.h:70-110), Euler1DFlux.c:19
// (euler1d.h:61-85).
// ---------------------------------------------------------------------------
// The two end interfaces (0 and N) of the line systems, a thread per pair of
// systems and end: WENO5 values on identity rows
// (Interp1PrimFifthOrderCRWENO.c:132-201 with the WENO5 weights at the ends).
// The raw values go to the case's `ends` table for the line solves, and, in
// paired mode their combination, to the interface arrays.  w: the six values at
// positions k-3 .. k+2.
template <int KIND>
__device__ __forceinline__ void recon_end(const CaseDev &C, int dir, long pair, int e, const double w[6]) {
  const SweepGeom &S = dir ? C.Sy : C.Sx;
  const int nv = C.G.nv, N = S.N, nl = S.nlines;
  const int q = (int)(pair % 2), v = (int)((pair / 2) % nv), l = (int)((pair / 2) / nv);
  const int k = e ? N : 0;
  const Global<double> *io = dir ? C.iy : C.ix;
  const long at = ((long)v * nl + l) * (N + 1) + k;
  double a, b, c, xl, xr;
  row_coeffs<KIND>(k, N, true, C.R, w[0], w[1], w[2], w[3], w[4], w[5], a, b, c, xl);
  row_coeffs<KIND>(k, N, false, C.R, w[0], w[1], w[2], w[3], w[4], w[5], a, b, c, xr);
  double *ends = C.ends + 4 * ((dir ? recon_pairs(C.Sx, nv) : 0) + pair);
  ends[e] = xl;
  ends[2 + e] = xr;
  if (C.paired) {
    io[q][at] = q ? 0.5 * (xl + xr) : 0.5 * (xr - xl);
  } else {
    io[2 * q][at] = xl;
    io[2 * q + 1][at] = xr;
  }
}

__host__ __device__ inline long end_items(const CaseDev &C) {
  return C.R.crweno && !C.R.characteristic
             ? 2 * (recon_pairs(C.Sx, C.G.nv) + (C.G.ndims == 2 ? recon_pairs(C.Sy, C.G.nv) : 0))
             : 0;
}

// item t of the ends; from_flux: the flux at the six positions is in memory,
// else it is formed here
__device__ __forceinline__ void recon_ends_item(const CaseDev &C, long t, int only, bool from_flux) {
  if (t >= end_items(C)) return;
  const int nv = C.G.nv;
  const long nx = 2 * recon_pairs(C.Sx, nv);
  const int dir = t < nx ? 0 : 1;
  const long pair = (dir ? t - nx : t) >> 1;
  const int e = (int)(t & 1), q = (int)(pair % 2), v = (int)((pair / 2) % nv), l = (int)((pair / 2) / nv);
  if (only && (dir != ((only >> 3) & 1) || q != ((only >> 2) & 1))) return;
  const SweepGeom &S = dir ? C.Sy : C.Sx;
  const long pl = S.plane, at = S.base + (long)l * S.line_stride + (e ? S.N : 0) - 3;
  const double *u = (dir ? C.UT : C.U) + at, *f = (dir ? C.flux_y : C.flux_x) + at;
  const int nf = C.model == 1 ? 3 : 4;
  double w[6];
  // three positions at a time, every load before the first is needed (with a branch
  // per position a wave took 17000 cycles, six round trips one after the other)
#pragma unroll
  for (int h = 0; h < 6; h += 3) {
    double c[3][4], x[3];
    const double *own = (from_flux && q ? f : u) + v * pl + h;
#pragma unroll
    for (int p = 0; p < 3; p++) {
      x[p] = own[p];
#pragma unroll
      for (int m = 0; m < 4; m++) c[p][m] = from_flux ? 0.0 : u[min(m, nf - 1) * pl + h + p];
    }
#pragma unroll
    for (int p = 0; p < 3; p++) {
      w[h + p] = x[p];
      if (from_flux) continue;
      double y = 0.0;
      point_flux(C.model, dir, C.P.gamma, nf + 1, [&](int m) { return m < nf ? c[p][m] : x[p]; },
                 [&](int m, double z) { y = m == (v < nf ? v : nf) ? z : y; });
      w[h + p] = q ? y : x[p];
    }
  }
  switch (C.R.kind) {
    case 1: recon_end<1>(C, dir, pair, e, w); break;
    case 2: recon_end<2>(C, dir, pair, e, w); break;
    case 3: recon_end<3>(C, dir, pair, e, w); break;
    default: recon_end<0>(C, dir, pair, e, w); break;
  }
}

// the end interfaces alone, from given arrays (the operators)
__global__ void __launch_bounds__(256) k_recon_ends(CASE_ARGS) {
  CASE_PREAMBLE
  if ((stage & 0xFF) < C.nstages) recon_ends_item(C, t, stage >> 8, true);
}

__host__ __device__ inline long flux_items(const CaseDev &C) {
  return (long)(C.Sx.N + 2 * C.Sx.g) * C.Sx.nlines +
         (C.G.ndims == 2 ? (long)(C.Sy.N + 2 * C.Sy.g) * C.Sy.nlines : 0);
}

// all: every component in its own plane, also where the reconstruction needs the
// velocity only
__device__ __forceinline__ void flux_item(const CaseDev &C, long t, bool all) {
  const long nX = (long)(C.Sx.N + 2 * C.Sx.g) * C.Sx.nlines;
  const long nY = (C.G.ndims == 2) ? (long)(C.Sy.N + 2 * C.Sy.g) * C.Sy.nlines : 0;
  if (t >= nX + nY) return;
  const int dir = t < nX ? 0 : 1;
  const SweepGeom &S = dir == 0 ? C.Sx : C.Sy;
  const long tt = dir == 0 ? t : t - nX;
  const double *q = dir == 0 ? C.U : C.UT;
  double *f = dir == 0 ? C.flux_x : C.flux_y;
  const int P = S.N + 2 * S.g;
  const int pos = (int)(tt % P) - S.g, l = (int)(tt / P);
  const long b = S.base + (long)l * S.line_stride + pos;
  const long pl = S.plane;
  const bool vn = C.vn_flux && !all;
  const int nf = C.model == 1 ? 3 : 4;
  point_flux(C.model, dir, C.P.gamma, vn ? nf : C.G.nv, [&](int m) { return q[m * pl + b]; },
             [&](int m, double x) { f[m * pl + b] = x; });
  if (vn) {
    const double rho = q[b], mom = q[(1 + dir) * pl + b];
    f[nf * pl + b] = C.model == 2 && rho == 0 ? 0 : mom / rho;
  }
  if (C.fuse_sp && pos >= 0 && pos <= S.N) {  // |v_n| at interface pos, between cells pos-1 and pos
    const double uLc[4] = {q[b - 1], q[pl + b - 1], q[2 * pl + b - 1], q[3 * pl + b - 1]};
    const double uRc[4] = {q[b], q[pl + b], q[2 * pl + b], q[3 * pl + b]};
    C.dsp[dir][(long)l * (S.N + 1) + pos] =
        dir == 0 ? ns2d_roe_dsp<0>(C.P.gamma, uLc, uRc) : ns2d_roe_dsp<1>(C.P.gamma, uLc, uRc);
  }
}

// What the line-system schemes need of the stage state before their solves:
// the viscous fluxes, the systems' end values and the cell fluxes, each in
// blocks of its own (the first two take longest).  One launch of a few
// microseconds' work costs as much again; with three, and the viscous fluxes on
// a second stream (whose fork and join cost 10 us a stage), 128 x 97 took 6.26 ms
// where it took 4.77, cavity 128 x 128 (k_weno's launch) 4.15 -> 2.54.  Small grids
// wait for the longest block's chain: with the loads of the viscous tiles and of
// the ends issued together a launch takes 11.4 -> 7.7 us (128 x 97).  Large ones
// are bound by HBM: seven waves a SIMD, which the viscous blocks' registers would
// not allow by themselves, 78 us at 1024 x 1024, six 81, five 85.
__global__ void __launch_bounds__(256, 7) k_flux(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage >= C.nstages) return;
  __shared__ Prims prims;
  const int bid = (int)blockIdx.x - first;
  const int nvis = viscous_blocks(C), nends = (int)((end_items(C) + TB - 1) / TB);
  if (bid < nvis) viscous_tile(C, bid, prims);
  else if (bid < nvis + nends) recon_ends_item(C, t - (long)nvis * TB, 0, false);
  else flux_item(C, t - (long)(nvis + nends) * TB, false);
}

// the cell fluxes alone, of any case (the operators)
__global__ void __launch_bounds__(256) k_flux_all(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage < C.nstages) flux_item(C, t, true);
}

// ---------------------------------------------------------------------------
// Characteristic CRWENO5: Interp1PrimFifthOrderCRWENOChar.c:96-280 with the
// reference's block solver (blocktridiagLU.c:159-180 and :279-301 on one
// process; _MatrixInvert_ etc., matops.h:16-130).  Each interface row ties
// the characteristic fields through L of the Roe average at that interface,
// so the unknowns are the physical interface values and every row is a block
// row.  L's species block is the identity, and the reference's dense n x n
// arithmetic then reduces exactly (up to the sign of zeros) to the flow block
// plus one scalar chain per species; both are computed here in the
// reference's operation order.
// ---------------------------------------------------------------------------

// block rows of every system at interface k of line l, one thread each, the
// line index fastest: a wave reads the same position of consecutive lines,
// contiguous in the other layout (the x sweep reads the transposed copy, the
// y sweep the natural one), and computes the flux there as k_flux does
template <int MODEL, int DIR, int KIND>
__device__ __forceinline__ void cwc_rows(const CaseDev &C, const SweepGeom &S, int l, int k, double *rows) {
  constexpr int NF = MODEL == 1 ? 3 : 4;
  const int nv = C.G.nv, nl = S.nlines, N = S.N;
  const double gam = C.P.gamma;
  // state at position pos of line l
  const double *q;
  long o0, ostr, pl;
  if (MODEL == 1) {
    q = C.U; o0 = S.base + (long)l * S.line_stride; ostr = 1; pl = S.plane;
  } else {
    const SweepGeom &O = DIR ? C.Sx : C.Sy;
    q = DIR ? C.U : C.UT; o0 = O.base + l; ostr = O.line_stride; pl = O.plane;
  }
  auto at = [&](int v, int pos) { return q[(long)v * pl + o0 + (long)pos * ostr]; };
  double L[NF][NF];
  if (MODEL == 1) {
    double a0, a1, a2;
    euler1d_roeavg(gam, at(0, k - 1), at(1, k - 1), at(2, k - 1), at(0, k), at(1, k), at(2, k), a0, a1, a2);
    Eig3 E;
    euler1d_eig(gam, a0, a1, a2, E);
#pragma unroll
    for (int i = 0; i < NF; i++)
#pragma unroll
      for (int j = 0; j < NF; j++) L[i][j] = E.L[i][j];
  } else {
    // the reference averages (k-1, k) for the left bias and (k, k-1) for the
    // right one; the Roe average is symmetric to the bit
    const double uLc[4] = {at(0, k - 1), at(1, k - 1), at(2, k - 1), at(3, k - 1)};
    const double uRc[4] = {at(0, k), at(1, k), at(2, k), at(3, k)};
    double ua[4], L4[4][4], R4[4][4];
    ns2d_roeavg(gam, uLc, uRc, ua);
    ns2d_eigvecs<DIR>(gam, ua, L4, R4);
#pragma unroll
    for (int i = 0; i < NF; i++)
#pragma unroll
      for (int j = 0; j < NF; j++) L[i][j] = L4[i][j];
  }
  const long vs = (long)nl * (N + 1), ii = (long)k * nl + l;
#pragma unroll
  for (int i = 0; i < NF; i++)
#pragma unroll
    for (int j = 0; j < NF; j++) rows[(long)(i * NF + j) * vs + ii] = L[i][j];
  const bool bnd = (k == 0 || k == N);
  // optimal weights: WENO5 at the physical ends, CRWENO5 inside
  // (WENOFifthOrderCalculateWeights.c:846-862)
  const double c1 = bnd ? 0.1 : 0.2, c2 = bnd ? 0.6 : 0.5, c3 = 0.3;
  const double s6 = 1.0 / 6.0, t3 = 1.0 / 3.0;
  const ReconParams &P = C.R;
  auto row = [&](int sys, int v, double m3, double m2, double m1, double p1, double p2) {
    double w1, w2, w3, f1, f2, f3, ca, cb, cc;
    if (P.no_limiting) { w1 = c1; w2 = c2; w3 = c3; }
    else weno_w<KIND>(c1, c2, c3, m3, m2, m1, p1, p2, P.eps, w1, w2, w3);
    if (bnd) {  // WENO5 row, B = L
      f1 = (2 * s6) * m3 - (7.0 * s6) * m2 + (11.0 * s6) * m1;
      f2 = (-s6) * m2 + (5.0 * s6) * m1 + (2 * s6) * p1;
      f3 = (2 * s6) * m1 + (5 * s6) * p1 - (s6)*p2;
      ca = 0.0; cb = 1.0; cc = 0.0;
    } else {
      f1 = (s6) * (m2 + 5 * m1);
      f2 = (s6) * (5 * m1 + p1);
      f3 = (s6) * (m1 + 5 * p1);
      const double wa = ((2 * t3) * w1 + (t3)*w2), wb = ((t3)*w1 + (2 * t3) * (w2 + w3)), wc = ((t3)*w3);
      const bool left = !(sys & 1);  // the right bias swaps the sub- and super-diagonal coefficients
      ca = left ? wa : wc;
      cb = wb;
      cc = left ? wc : wa;
    }
    const long b = (long)(NF * NF + (sys * nv + v) * 4) * vs + ii;
    rows[b] = ca;
    rows[b + vs] = cb;
    rows[b + 2 * vs] = cc;
    rows[b + 3 * vs] = w1 * f1 + w2 * f2 + w3 * f3;
  };
  // flow state, flux and characteristic values at k-3 .. k+2
  double cu[6][NF], cf[6][NF], vn[6];
#pragma unroll
  for (int p = 0; p < 6; p++) {
    const int pos = k - 3 + p;
    double x[NF], fx[NF];
#pragma unroll
    for (int j = 0; j < NF; j++) x[j] = at(j, pos);
    if (MODEL == 1) {
      const double rho = x[0], v = x[1] / rho, e = x[2], P_ = (e - 0.5 * rho * v * v) * (gam - 1.0);
      fx[0] = rho * v;
      fx[1] = rho * v * v + P_;
      fx[2] = (e + P_) * v;
      vn[p] = v;
    } else {
      const double rho = x[0], vx = (rho == 0) ? 0 : x[1] / rho, vy = (rho == 0) ? 0 : x[2] / rho, e = x[3];
      const double vsq = (vx * vx) + (vy * vy), P_ = (e - 0.5 * rho * vsq) * (gam - 1.0);
      const double v = DIR == 0 ? vx : vy;
      fx[0] = rho * v;
      if (DIR == 0) { fx[1] = rho * vx * vx + P_; fx[2] = rho * vx * vy; }
      else { fx[1] = rho * vy * vx; fx[2] = rho * vy * vy + P_; }
      fx[NF - 1] = (e + P_) * v;
      vn[p] = v;
    }
#pragma unroll
    for (int v = 0; v < NF; v++) {
      double au = L[v][0] * x[0], af = L[v][0] * fx[0];
#pragma unroll
      for (int j = 1; j < NF; j++) {
        au = au + L[v][j] * x[j];
        af = af + L[v][j] * fx[j];
      }
      cu[p][v] = au;
      cf[p][v] = af;
    }
  }
#pragma unroll
  for (int v = 0; v < NF; v++) {
    row(0, v, cu[0][v], cu[1][v], cu[2][v], cu[3][v], cu[4][v]);
    row(1, v, cu[5][v], cu[4][v], cu[3][v], cu[2][v], cu[1][v]);
    row(2, v, cf[0][v], cf[1][v], cf[2][v], cf[3][v], cf[4][v]);
    row(3, v, cf[5][v], cf[4][v], cf[3][v], cf[2][v], cf[1][v]);
  }
  for (int m = NF; m < nv; m++) {  // passive scalars: identity rows, flux vn u_m
    double x[6], fx[6];
#pragma unroll
    for (int p = 0; p < 6; p++) {
      x[p] = at(m, k - 3 + p);
      fx[p] = vn[p] * x[p];
    }
    row(0, m, x[0], x[1], x[2], x[3], x[4]);
    row(1, m, x[5], x[4], x[3], x[2], x[1]);
    row(2, m, fx[0], fx[1], fx[2], fx[3], fx[4]);
    row(3, m, fx[5], fx[4], fx[3], fx[2], fx[1]);
  }
}

__global__ void __launch_bounds__(256) k_cw_rows(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage >= C.nstages) return;
  const long nX = (long)(C.Sx.N + 1) * C.Sx.nlines;
  const long nY = (C.G.ndims == 2) ? (long)(C.Sy.N + 1) * C.Sy.nlines : 0;
  if (t >= nX + nY) return;
  const int dir = t < nX ? 0 : 1;
  const SweepGeom &S = dir ? C.Sy : C.Sx;
  const long u = dir ? t - nX : t;
  const int l = (int)(u % S.nlines), k = (int)(u / S.nlines);
  double *rows = C.cwr[dir];
#define CWROWS(KIND)                                                \
  (C.model == 1 ? cwc_rows<1, 0, KIND>(C, S, l, k, rows)           \
                : (dir ? cwc_rows<2, 1, KIND>(C, S, l, k, rows)    \
                       : cwc_rows<2, 0, KIND>(C, S, l, k, rows)))
  switch (C.R.kind) {
    case 1: CWROWS(1); break;
    case 2: CWROWS(2); break;
    case 3: CWROWS(3); break;
    default: CWROWS(0); break;
  }
#undef CWROWS
}

// A species chain (chain >= 1): the scalar chain of the same arithmetic as the
// flow block's, for species NF + chain - 1.
// Segments of a block chain: rows 1..N of the forward elimination split into
// `segs` runs of cw_seg_rows rows, each run owned by a lane (species) or a
// quad of lanes (flow) of the same wave.  A run starts from an estimate of
// the state entering it (its first row taken as if it were the system's
// first), runs the reference's row steps, and hands its exit state on; a run
// whose entry differs from its predecessor's exit runs again from that exit
// until a row reproduces, bit for bit, what the previous pass stored there
// (the chain depends on the past only through that row's stored values, so
// every later row would repeat too).  Run 0 starts from row 0 exactly, so
// the fixed point is the sequential chain's, bit for bit; the recurrences
// contract, so a run of a few dozen rows forgets its estimate and one
// correcting pass usually suffices.  The back substitution is relayed the
// same way from the top.  segs = 1 is the sequential chain.  After relay pass
// p, runs 0 .. p+1 hold the sequential chain (run p+1 has started from run
// p's exact exit), so segs - 1 passes always suffice and the loops' bound of
// segs + 1 passes is never what ends them.
#ifndef PIAFS_CW_RMIN
#define PIAFS_CW_RMIN 128
#endif
#ifndef PIAFS_CW_LANES
#define PIAFS_CW_LANES 65536
#endif
__host__ __device__ inline int cw_segs(const SweepGeom &S, int nv, int nf) {
  const long lanes = 4L * S.nlines * (4 + nv - nf);  // lanes of the sweep's chains unsegmented
  int s = 1;
  while (s < 16 && 2 * s * PIAFS_CW_RMIN <= S.N + 1 && 2 * s * lanes <= PIAFS_CW_LANES) s <<= 1;
  return s;
}
__host__ __device__ inline int cw_seg_rows(int N, int segs) { return (N + segs - 1) / segs; }

__device__ __forceinline__ void cwc_species(const CaseDev &C, const SweepGeom &S, int dir, int l, int sys,
                                           int chain, int NF, int seg, int segs) {
  const int nv = C.G.nv, nl = S.nlines, N = S.N;
  const long vs = (long)nl * (N + 1);
  const long bs = 4L * nl * (N + 1), bb = (long)sys * (N + 1) * nl + l;
  const double *rows = C.cwr[dir];
  double *back = C.cwb[dir];
  double *out = (dir ? C.iy : C.ix)[sys];
  auto rf = [&](int f, int k) { return rows[(long)f * vs + (long)k * nl + l]; };
  auto bk = [&](int f, int k) -> double & { return back[(long)f * bs + bb + (long)k * nl]; };
  auto coef = [&](int v, int which, int k) { return rf(NF * NF + (sys * nv + v) * 4 + which, k); };
  const int m = NF + chain - 1, f0 = 2 * NF * NF + NF + 3 * (chain - 1);
  const int R = cw_seg_rows(N, segs);
  const int k0 = 1 + seg * R, k1 = min(N + 1, k0 + R);  // forward rows of this run
  const bool has = k0 < k1;
  const int lane = threadIdx.x & 63;
  // forward: rows k0..k1-1, row k storing (1/b'_{k-1}, c_{k-1}, x'_{k-1}) at k-1
  double bp, xp, cprev;
  {
    const int ks = seg == 0 ? 0 : (has ? k0 - 1 : 0);
    bp = coef(m, 1, ks);
    xp = coef(m, 3, ks);
    cprev = coef(m, 2, ks);
  }
  // one pass from the entry (bp, xp); early: stop where a row repeats its stored values
  auto forward = [&](bool early) {
    double a = has ? coef(m, 0, k0) : 0.0, b = has ? coef(m, 1, k0) : 0.0, c = has ? coef(m, 2, k0) : 0.0,
           F = has ? coef(m, 3, k0) : 0.0;
    // what the previous pass stored at k-1, loaded one row ahead like the coefficients
    double srb = early && has ? bk(f0, k0 - 1) : 0.0, sxp = early && has ? bk(f0 + 2, k0 - 1) : 0.0;
    for (int k = k0; k < k1; k++) {
      const double na = k + 1 < k1 ? coef(m, 0, k + 1) : 0.0, nb = k + 1 < k1 ? coef(m, 1, k + 1) : 0.0,
                   nc = k + 1 < k1 ? coef(m, 2, k + 1) : 0.0, nF = k + 1 < k1 ? coef(m, 3, k + 1) : 0.0;
      const double crb = srb, cxp = sxp;
      if (early && k + 1 < k1) {
        srb = bk(f0, k);
        sxp = bk(f0 + 2, k);
      }
      const double rb = 1.0 / bp, fac = a * rb;
      if (early && __double_as_longlong(rb) == __double_as_longlong(crb) &&
          __double_as_longlong(xp) == __double_as_longlong(cxp))
        return false;  // this row and every later one as stored
      bk(f0, k - 1) = rb;
      bk(f0 + 1, k - 1) = cprev;
      bk(f0 + 2, k - 1) = xp;
      bp = b - fac * cprev;
      xp = F - fac * xp;
      cprev = c;
      a = na; b = nb; c = nc; F = nF;
    }
    return true;
  };
  forward(false);
  double ebp = bp, exp_ = xp;  // exit state
  double nbp = bp, nxp = xp;   // the entry this run last started from (set below)
  {
    // the entry of the first pass, for the comparison with the predecessor's exit
    const int ks = seg == 0 ? 0 : (has ? k0 - 1 : 0);
    nbp = coef(m, 1, ks);
    nxp = coef(m, 3, ks);
    if (seg == 0) {  // run 0 starts at row 0: b'_0 = b_0, x'_0 = F_0
      nbp = coef(m, 1, 0);
      nxp = coef(m, 3, 0);
    }
  }
  for (int pass = 0;; pass++) {
    const double pbp = __shfl(ebp, lane - 1), pxp = __shfl(exp_, lane - 1);
    const bool changed = seg > 0 && (__double_as_longlong(pbp) != __double_as_longlong(nbp) ||
                                     __double_as_longlong(pxp) != __double_as_longlong(nxp));
    if (!__any(changed) || pass > segs) break;
    if (changed) {
      nbp = pbp;
      nxp = pxp;
      if (!has) {
        ebp = pbp;
        exp_ = pxp;
      } else {
        bp = pbp;
        xp = pxp;
        cprev = coef(m, 2, k0 - 1);
        if (forward(true)) {
          ebp = bp;
          exp_ = xp;
        }
      }
    }
  }
  // back substitution: rows k1-2 .. k0-1 of this run (the top run also row N),
  // entering from the run above
  const long ob = ((long)m * nl + l) * (N + 1);
  const bool top = k1 == N + 1 && (has || N == 0);
  double xin = 0.0;  // x of the row above this run's rows
  if (top) {
    xin = (1.0 / ebp) * exp_;
    out[ob + N] = xin;
  }
  auto backward = [&](double x, bool early) {
    int k = k1 - 2;
    if (k < k0 - 1) return;
    // each row's values loaded one row ahead
    double nrb = bk(f0, k), ncp = bk(f0 + 1, k), nxq = bk(f0 + 2, k), nso = early ? out[ob + k] : 0.0;
    for (; k >= k0 - 1; k--) {
      const double rb = nrb, c = ncp, xq = nxq, so = nso;
      if (k > k0 - 1) {
        nrb = bk(f0, k - 1);
        ncp = bk(f0 + 1, k - 1);
        nxq = bk(f0 + 2, k - 1);
        if (early) nso = out[ob + k - 1];
      }
      x = rb * (xq - c * x);
      if (early && __double_as_longlong(x) == __double_as_longlong(so)) return;
      out[ob + k] = x;
    }
  };
  double xs = xin;  // the entry the last pass started from
  if (has) backward(xin, false);
  for (int pass = 0;; pass++) {
    // the exit of a run is the x of its lowest row; an empty run passes its entry on
    const double mine = has ? out[ob + k0 - 1] : xs;
    const double above = __shfl(mine, lane + 1);
    const bool last = seg == segs - 1 || top;
    const bool changed = !last && __double_as_longlong(above) != __double_as_longlong(xs);
    if (!__any(changed) || pass > segs) break;
    if (changed) {
      xs = above;
      if (has) backward(above, true);
    }
  }
}

// The flow block chain of one system of one line (blocktridiagLU.c:159-301
// with the blocks inverted by _MatrixInvert_, matops.h:96-130: Gauss-Jordan
// without pivoting) on the four lanes of a quad: lane r < NF holds row r of
// every NF x NF block and row r of the vectors (x', the solution); lane 3 in
// 1D only takes part in the exchanges.  Rows move between the lanes by DPP
// quad permutations (no LDS), and each lane keeps whole copies of the blocks
// it multiplies by (the inverse, C_{k-1}).  Every entry goes through the
// reference's operations in its order: a step of the inverse updates only
// rows that the rows it reads do not depend on.  All four lanes execute every
// exchange (none sits under a lane-dependent branch).
template <int SRC>
__device__ __forceinline__ double quad_get(double v) {
  constexpr int ctrl = SRC | (SRC << 2) | (SRC << 4) | (SRC << 6);  // quad_perm [SRC, SRC, SRC, SRC]
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b & 0xffffffffLL), ctrl, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)((unsigned long long)b >> 32), ctrl, 0xF, 0xF, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ double qget(double v, int src) {  // src is a constant after unrolling
  switch (src) {
    case 0: return quad_get<0>(v);
    case 1: return quad_get<1>(v);
    case 2: return quad_get<2>(v);
    default: return quad_get<3>(v);
  }
}

// inverse of the block whose row ri this lane holds in bp; every lane gets the
// whole inverse.  Its divisions (elimination factors and back substitution)
// take wdiv: the IEEE quotient's bits for the blocks' operands, except that an
// exactly zero numerator -0 over a positive pivot gives +0; the inverse's
// entries are never divisors, so no nonzero value downstream changes.
#ifndef PIAFS_CW_FAST_INV
#define PIAFS_CW_FAST_INV 1
#endif
#if PIAFS_CW_FAST_INV
#define CW_DIV(n, d) wdiv(n, d)
#else
#define CW_DIV(n, d) ((n) / (d))
#endif
template <int NF>
__device__ __forceinline__ void cw_inv_quad(const double (&bp)[NF], int ri, double (&Bi)[NF][NF]) {
  double ac[NF], bb[NF];
#pragma unroll
  for (int j = 0; j < NF; j++) {
    ac[j] = bp[j];
    bb[j] = (ri == j) ? 1.0 : 0.0;
  }
#pragma unroll
  for (int i = 0; i < NF - 1; i++) {
    double pa[NF], pb[NF];
#pragma unroll
    for (int k = 0; k < NF; k++) {
      pa[k] = qget(ac[k], i);
      pb[k] = qget(bb[k], i);
    }
    if (ri > i) {
      const double f = CW_DIV(ac[i], pa[i]);
#pragma unroll
      for (int k = i + 1; k < NF; k++) ac[k] -= (f * pa[k]);
#pragma unroll
      for (int k = 0; k < NF; k++)
        if (k < ri) bb[k] -= (f * pb[k]);
    }
  }
#pragma unroll
  for (int i = NF - 1; i >= 0; i--) {
    if (ri == i) {
#pragma unroll
      for (int k = 0; k < NF; k++) {
        double sum = 0.0;
#pragma unroll
        for (int j = i + 1; j < NF; j++) sum += (ac[j] * Bi[j][k]);
        bb[k] = CW_DIV(bb[k] - sum, ac[i]);
      }
    }
#pragma unroll
    for (int k = 0; k < NF; k++) Bi[i][k] = qget(bb[k], i);
  }
}

// all four lanes of the quad hold p
__device__ __forceinline__ bool quad_all(bool p) {
  const double d = p ? 1.0 : 0.0;
  return quad_get<0>(d) * quad_get<1>(d) * quad_get<2>(d) * quad_get<3>(d) == 1.0;
}

template <int NF>
__device__ __forceinline__ void cwc_flow_quad(const CaseDev &C, const SweepGeom &S, int dir, int l, int sys, int e,
                                              int seg, int segs) {
  const int nv = C.G.nv, nl = S.nlines, N = S.N;
  const bool act = e < NF;
  const int ri = act ? e : NF - 1;  // the spare lane of a 1D quad reads row NF-1 and stores nothing
  const long vs = (long)nl * (N + 1);
  const long bs = 4L * nl * (N + 1), bb = (long)sys * (N + 1) * nl + l;
  const double *rows = C.cwr[dir];
  double *back = C.cwb[dir];
  double *out = (dir ? C.iy : C.ix)[sys];
  auto rf = [&](int f, int k) { return rows[(long)f * vs + (long)k * nl + l]; };
  auto bk = [&](int f, int k) -> double & { return back[(long)f * bs + bb + (long)k * nl]; };
  auto coef = [&](int which, int k) { return rf(NF * NF + (sys * nv + ri) * 4 + which, k); };
  const int R = cw_seg_rows(N, segs);
  const int k0 = 1 + seg * R, k1 = min(N + 1, k0 + R);  // forward rows of this run
  const bool has = k0 < k1;
  const int lane = threadIdx.x & 63;
  // this lane's row of the blocks of row k: A = a L, B = b L, C = c L, and F
  auto row = [&](int k, double (&A)[NF], double (&Bm)[NF], double (&Cm)[NF], double &F) {
    const double a = coef(0, k), b = coef(1, k), c = coef(2, k);
    F = coef(3, k);
#pragma unroll
    for (int j = 0; j < NF; j++) {
      const double Lj = rf(NF * ri + j, k);
      A[j] = a * Lj;
      Bm[j] = b * Lj;
      Cm[j] = c * Lj;
    }
  };
  // state after row k-1: row ri of B', row ri of C, component ri of x'
  double bp[NF], cprev[NF], xp;
  auto first = [&](int k) {  // row k as the first row of the chain
    double A[NF], Bm[NF], Cm[NF], F;
    row(k, A, Bm, Cm, F);
    xp = F;
#pragma unroll
    for (int j = 0; j < NF; j++) {
      bp[j] = Bm[j];
      cprev[j] = Cm[j];
    }
  };
  // one pass over rows k0..k1-1 (row k stores the inverse of B'_{k-1}, C_{k-1}
  // and x'_{k-1} at k-1); early: stop where a row repeats what is stored
  auto forward = [&](bool early) {
    // row k+1's coefficients and what the previous pass stored at k are loaded one row ahead
    double na = 0.0, nb = 0.0, nc = 0.0, nF = 0.0, nL[NF], sBi[NF], sxp = 0.0;
#pragma unroll
    for (int j = 0; j < NF; j++) nL[j] = sBi[j] = 0.0;
    auto load = [&](int k) {
      na = coef(0, k);
      nb = coef(1, k);
      nc = coef(2, k);
      nF = coef(3, k);
#pragma unroll
      for (int j = 0; j < NF; j++) nL[j] = rf(NF * ri + j, k);
    };
    auto load_stored = [&](int k) {
#pragma unroll
      for (int j = 0; j < NF; j++) sBi[j] = bk(NF * ri + j, k);
      sxp = bk(2 * NF * NF + ri, k);
    };
    if (has) load(k0);
    if (early && has) load_stored(k0 - 1);
    for (int k = k0; k < k1; k++) {
      double A[NF], Bm[NF], Cm[NF], cBi[NF];
      const double F = nF, cxp = sxp;
#pragma unroll
      for (int j = 0; j < NF; j++) {
        A[j] = na * nL[j];
        Bm[j] = nb * nL[j];
        Cm[j] = nc * nL[j];
        cBi[j] = sBi[j];
      }
      if (k + 1 < k1) {
        load(k + 1);
        if (early) load_stored(k);
      }
      double Bi[NF][NF];
      cw_inv_quad<NF>(bp, ri, Bi);
      if (early) {
        bool same = __double_as_longlong(xp) == __double_as_longlong(cxp);
#pragma unroll
        for (int j = 0; j < NF; j++) same = same && __double_as_longlong(Bi[ri][j]) == __double_as_longlong(cBi[j]);
        if (quad_all(same || !act)) return false;  // this row and every later one as stored
      }
      double fac[NF];
#pragma unroll
      for (int j = 0; j < NF; j++) {
        double acc = 0;
#pragma unroll
        for (int q = 0; q < NF; q++) acc += (A[q] * Bi[q][j]);
        fac[j] = acc;
      }
      if (act) {
#pragma unroll
        for (int j = 0; j < NF; j++) {
          bk(NF * ri + j, k - 1) = Bi[ri][j];
          bk(NF * NF + NF * ri + j, k - 1) = cprev[j];
        }
        bk(2 * NF * NF + ri, k - 1) = xp;
      }
      double cpf[NF][NF], xpf[NF];
#pragma unroll
      for (int q = 0; q < NF; q++) {
        xpf[q] = qget(xp, q);
#pragma unroll
        for (int j = 0; j < NF; j++) cpf[q][j] = qget(cprev[j], q);
      }
      double xn = F;
#pragma unroll
      for (int j = 0; j < NF; j++) {
        double bn = Bm[j];
#pragma unroll
        for (int q = 0; q < NF; q++) bn -= (fac[q] * cpf[q][j]);
        bp[j] = bn;
      }
#pragma unroll
      for (int q = 0; q < NF; q++) xn -= (fac[q] * xpf[q]);
      xp = xn;
#pragma unroll
      for (int j = 0; j < NF; j++) cprev[j] = Cm[j];
    }
    return true;
  };
  // run 0 starts at row 0 exactly; the others from their first row's predecessor taken as a first row
  first(seg == 0 || !has ? 0 : k0 - 1);
  double nbp[NF], nxp = xp;  // the entry this run last started from
#pragma unroll
  for (int j = 0; j < NF; j++) nbp[j] = bp[j];
  if (has) forward(false);
  double ebp[NF], exq = xp;  // exit state
#pragma unroll
  for (int j = 0; j < NF; j++) ebp[j] = bp[j];
  for (int pass = 0;; pass++) {
    double pbp[NF];
    bool changed = false;
#pragma unroll
    for (int j = 0; j < NF; j++) {
      pbp[j] = __shfl(ebp[j], lane - 4);
      changed = changed || __double_as_longlong(pbp[j]) != __double_as_longlong(nbp[j]);
    }
    const double pxp = __shfl(exq, lane - 4);
    changed = seg > 0 && (changed || __double_as_longlong(pxp) != __double_as_longlong(nxp));
    changed = !quad_all(!changed);  // a quad moves as one
    if (!__any(changed) || pass > segs) break;
    if (changed) {
#pragma unroll
      for (int j = 0; j < NF; j++) nbp[j] = bp[j] = pbp[j];
      nxp = xp = pxp;
      if (!has) {
#pragma unroll
        for (int j = 0; j < NF; j++) ebp[j] = pbp[j];
        exq = pxp;
      } else {
        double A[NF], Bm[NF], Cm[NF], F;
        row(k0 - 1, A, Bm, Cm, F);
#pragma unroll
        for (int j = 0; j < NF; j++) cprev[j] = Cm[j];
        if (forward(true)) {
#pragma unroll
          for (int j = 0; j < NF; j++) ebp[j] = bp[j];
          exq = xp;
        }
      }
    }
  }
  // back substitution x_k = binv_k (x'_k - C_k x_{k+1}): rows k1-2 .. k0-1 of
  // this run, the top run also row N, entering from the run above
  const long ob = ((long)ri * nl + l) * (N + 1);
  const bool top = k1 == N + 1 && (has || N == 0);
  double xin = 0.0;
  if (top) {
    double Bi[NF][NF], xpf[NF];
#pragma unroll
    for (int j = 0; j < NF; j++) bp[j] = ebp[j];
    cw_inv_quad<NF>(bp, ri, Bi);
#pragma unroll
    for (int q = 0; q < NF; q++) xpf[q] = qget(exq, q);
    double x = 0;
#pragma unroll
    for (int j = 0; j < NF; j++) x += (Bi[ri][j] * xpf[j]);
    if (act) out[ob + N] = x;
    xin = x;
  }
  auto backward = [&](double x, bool early) {
    int k = k1 - 2;
    if (k < k0 - 1) return;
    // each row's values loaded one row ahead
    double nbi[NF], ncp[NF], nxq = 0.0, nso = 0.0;
    auto load_back = [&](int k) {
#pragma unroll
      for (int j = 0; j < NF; j++) {
        nbi[j] = bk(NF * ri + j, k);
        ncp[j] = bk(NF * NF + NF * ri + j, k);
      }
      nxq = bk(2 * NF * NF + ri, k);
      if (early) nso = out[ob + k];
    };
    load_back(k);
    for (; k >= k0 - 1; k--) {
      double bi[NF], cp[NF], xf[NF], yf[NF];
      const double so = nso;
#pragma unroll
      for (int j = 0; j < NF; j++) {
        bi[j] = nbi[j];
        cp[j] = ncp[j];
        xf[j] = qget(x, j);
      }
      double y = nxq;
      if (k > k0 - 1) load_back(k - 1);
#pragma unroll
      for (int j = 0; j < NF; j++) y -= (cp[j] * xf[j]);
#pragma unroll
      for (int j = 0; j < NF; j++) yf[j] = qget(y, j);
      double xn = 0;
#pragma unroll
      for (int j = 0; j < NF; j++) xn += (bi[j] * yf[j]);
      x = xn;
      if (early && quad_all(!act || __double_as_longlong(x) == __double_as_longlong(so))) return;
      if (act) out[ob + k] = x;
    }
  };
  double xs = xin;  // the entry the last pass started from
  if (has) backward(xin, false);
  for (int pass = 0;; pass++) {
    const double mine = has ? out[ob + k0 - 1] : xs;  // this run's exit: the x of its lowest row
    const double above = __shfl(mine, lane + 4);
    const bool last = seg == segs - 1 || top;
    bool changed = !last && __double_as_longlong(above) != __double_as_longlong(xs);
    changed = !quad_all(!changed);
    if (!__any(changed) || pass > segs) break;
    if (changed) {
      xs = above;
      if (has) backward(above, true);
    }
  }
}

// Work items of a sweep: the flow chains first (a quad of lanes per run of a
// system; (run, system, line) with the run fastest), then one item per run of
// each species chain ((run, chain, system, line), the run fastest), so that
// the runs of a chain are neighbouring lanes of one wave.  The y sweep starts
// on a 64-item boundary, which keeps every quad of a flow chain on one quad
// of a wave.
__host__ __device__ inline int cw_flow_lanes(int) { return 4; }
__host__ __device__ inline long cw_items(const SweepGeom &S, int nv, int nf) {
  return 4L * S.nlines * cw_segs(S, nv, nf) * (cw_flow_lanes(nf) + nv - nf);
}
__host__ __device__ inline long cw_x_span(const CaseDev &c, int nf) {
  const long nX = cw_items(c.Sx, c.G.nv, nf);
  return c.G.ndims == 2 ? (nX + 63) & ~63L : nX;
}

#ifndef PIAFS_CWSOLVE_MINB
#define PIAFS_CWSOLVE_MINB 1
#endif
__global__ void __launch_bounds__(256, PIAFS_CWSOLVE_MINB) k_cw_solve(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage >= C.nstages) return;
  const int nv = C.G.nv, nf = C.model == 1 ? 3 : 4;
  const long nX = cw_items(C.Sx, nv, nf), nXs = cw_x_span(C, nf);
  const long nY = (C.G.ndims == 2) ? cw_items(C.Sy, nv, nf) : 0;
  if (t >= nXs + nY || (t >= nX && t < nXs)) return;
  const int dir = t < nXs ? 0 : 1;
  const SweepGeom &S = dir ? C.Sy : C.Sx;
  const long u = dir ? t - nXs : t;
  const int segs = cw_segs(S, nv, nf);
  const long nl = S.nlines, nflow = 4L * nl * cw_flow_lanes(nf) * segs;
  if (u < nflow) {
    const long quad = u >> 2, grp = quad / segs;
    const int seg = (int)(quad % segs);
    if (nf == 4) cwc_flow_quad<4>(C, S, dir, (int)(grp % nl), (int)(grp / nl), (int)(u & 3), seg, segs);
    else cwc_flow_quad<3>(C, S, dir, (int)(grp % nl), (int)(grp / nl), (int)(u & 3), seg, segs);
    return;
  }
  const long v = u - nflow, per = 4L * nl;
  const long ch = v / segs;
  const int seg = (int)(v % segs);
  const int chain = 1 + (int)(ch / per), sys = (int)((ch % per) / nl), l = (int)(ch % nl);
  cwc_species(C, S, dir, l, sys, chain, nf, seg, segs);
}

// ---------------------------------------------------------------------------
// Component-wise reconstruction of lines longer than one team covers
// (SweepGeom::longl).  k_lrows assembles every row of every system, end rows
// included, one thread per (system, interface), into the sweep's scratch,
// system by system ([A|B|C|X][system][interface]).  k_lsolve gives each pair
// of systems (uL and uR, or fL and fR of one line and variable) a block, whose
// 256 lanes walk the line window by window (kMaxRows rows per lane, 4096 rows
// a window): the forward elimination of each window (team_forward) starts
// from the exact pivot, super-diagonal and x' of the previous window's last
// row and stores b' and x'; the back substitution (team_backward) then runs
// the windows from the last, each from the exact solution of the row after
// it.  Every row goes through the reference's arithmetic (tridiagLU.c:133-150,
// :243-255, over rows 0..N with identity end rows), so the result is the
// sequential sweep's bit for bit.  The block then writes the interface arrays
// as the team kernels do.
// ---------------------------------------------------------------------------
__host__ __device__ inline long long_rows(const SweepGeom &S, int nv) {
  return S.longl ? (long)(S.N + 1) * S.nlines * nv * 4 : 0;
}

template <int KIND>
__device__ __forceinline__ void lrow_at(const CaseDev &C, int dir, long t) {
  const SweepGeom &S = dir ? C.Sy : C.Sx;
  const int nv = C.G.nv, N = S.N;
  const long ns4 = (long)S.nlines * nv * 4;
  const long sys = t / (N + 1);
  const int k = (int)(t % (N + 1));
  const int r = (int)(sys % 4), v = (int)((sys / 4) % nv), l = (int)(sys / 4 / nv);
  const double *src = (r < 2 ? (dir ? C.UT : C.U) : (dir ? C.flux_y : C.flux_x)) + (long)v * S.plane + S.base +
                      (long)l * S.line_stride;
  double a, b, c, x;
  row_coeffs<KIND>(k, N, !(r & 1), C.R, src[k - 3], src[k - 2], src[k - 1], src[k], src[k + 1], src[k + 2], a,
                       b, c, x);
  double *L = C.lrow[dir];
  const long f = (long)(N + 1) * ns4, o = sys * (N + 1) + k;
  L[o] = a;
  L[f + o] = b;
  L[2 * f + o] = c;
  L[3 * f + o] = x;
}

__global__ void __launch_bounds__(256) k_lrows(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage >= C.nstages) return;
  const long nX = long_rows(C.Sx, C.G.nv), nY = C.G.ndims == 2 ? long_rows(C.Sy, C.G.nv) : 0;
  if (t >= nX + nY) return;
  const int dir = t < nX ? 0 : 1;
  const long tt = dir ? t - nX : t;
  switch (C.R.kind) {
    case 1: lrow_at<1>(C, dir, tt); break;
    case 2: lrow_at<2>(C, dir, tt); break;
    case 3: lrow_at<3>(C, dir, tt); break;
    default: lrow_at<0>(C, dir, tt); break;
  }
}

// pairs of systems of the long sweeps, one block each
__host__ __device__ inline long long_pairs(const SweepGeom &S, int nv) {
  return S.longl ? (long)S.nlines * nv * 2 : 0;
}

// One system of a long line, rows 0..N of the scratch (A, B, C, X at
// interface k: L[arr*f + k]): rows 1..N-1 solved in windows of kLongWin
// rows, the identity rows 0 and N holding the end values.  On exit X holds
// the solution at every row.
constexpr int kLongTeam = 256, kLongWin = kLongTeam * kMaxRows;
__device__ void long_system(double *A, double *B, double *Cc, double *X, int N, double *red, double *carry,
                            bool plain_start, bool &zp) {
  const int lane = threadIdx.x;
  const int nwin = (N - 1 + kLongWin - 1) / kLongWin;  // interior rows 1..N-1
  auto window_rows = [&](int w, int &lo, int &n) {
    lo = 1 + w * kLongWin + lane * kMaxRows;
    n = N - lo;
    n = n < 0 ? 0 : (n > kMaxRows ? kMaxRows : n);
  };
  // forward: window w enters with the exact b', c and x' of the row before it
  double bfirst = 1.0, cfirst = 0.0, xfirst = X[0];  // row 0: identity, x' = its value
  for (int w = 0; w < nwin; w++) {
    int lo, n;
    window_rows(w, lo, n);
    double a[kMaxRows], b[kMaxRows], c[kMaxRows], x[kMaxRows], fk[kMaxRows];
#pragma unroll
    for (int i = 0; i < kMaxRows; i++) {
      const bool in = i < n;
      a[i] = in ? A[lo + i] : 0.0;
      b[i] = in ? B[lo + i] : 1.0;
      c[i] = in ? Cc[lo + i] : 0.0;
      x[i] = in ? X[lo + i] : 0.0;
    }
    team_forward<kMaxRows>(a, b, c, x, fk, n, lane, kLongTeam, bfirst, cfirst, xfirst, red, plain_start, zp);
#pragma unroll
    for (int i = 0; i < kMaxRows; i++)
      if (i < n) {
        B[lo + i] = b[i];
        X[lo + i] = x[i];
      }
    // the window's last row, from the lane that holds it, for the next window
    const int last = (w + 1) * kLongWin < N - 1 ? (w + 1) * kLongWin : N - 1;  // row index
    if (n > 0 && lo + n - 1 == last) {
      carry[0] = b[n - 1];
      carry[1] = c[n - 1];
      carry[2] = x[n - 1];
    }
    __syncthreads();
    bfirst = carry[0];
    cfirst = carry[1];
    xfirst = carry[2];
    __syncthreads();
  }
  // back substitution: window w ends at the row whose solution the window
  // after it (or row N, an identity row) has fixed
  double xlast = X[N];
  for (int w = nwin - 1; w >= 0; w--) {
    int lo, n;
    window_rows(w, lo, n);
    double b[kMaxRows], c[kMaxRows], x[kMaxRows], wk[kMaxRows];
#pragma unroll
    for (int i = 0; i < kMaxRows; i++) {
      const bool in = i < n;
      b[i] = in ? B[lo + i] : 1.0;
      c[i] = in ? Cc[lo + i] : 0.0;
      x[i] = in ? X[lo + i] : 0.0;
    }
    const int last = (w + 1) * kLongWin < N - 1 ? (w + 1) * kLongWin : N - 1;
    const bool is_last = n > 0 && lo + n - 1 == last;
    team_backward<kMaxRows>(b, c, x, wk, n, lane, kLongTeam, is_last, xlast, red, plain_start);
#pragma unroll
    for (int i = 0; i < kMaxRows; i++)
      if (i < n) X[lo + i] = x[i];
    if (lane == 0) carry[0] = x[0];  // the window's first row
    __syncthreads();
    xlast = carry[0];
    __syncthreads();
  }
}

__global__ void __launch_bounds__(kLongTeam) k_lsolve(CASE_ARGS) {
  CASE_PREAMBLE
  (void)t;
  if (stage >= C.nstages) return;
  __shared__ double red[16];
  __shared__ double carry[3];
  const int nv = C.G.nv;
  const long nX = long_pairs(C.Sx, nv);
  const long nY = C.G.ndims == 2 ? long_pairs(C.Sy, nv) : 0;
  const long pair = (int)blockIdx.x - first;
  if (pair >= nX + nY) return;  // uniform over the block
  const int dir = pair < nX ? 0 : 1;
  const long p = dir ? pair - nX : pair;  // (line*nv + var)*2 + q
  const SweepGeom &S = dir ? C.Sy : C.Sx;
  const int N = S.N, q = (int)(p % 2);
  const long lv = p / 2;  // line*nv + var
  const int v = (int)(lv % nv), l = (int)(lv / nv);
  const long ns4 = (long)S.nlines * nv * 4, f = (long)(N + 1) * ns4;
  double *L = C.lrow[dir];
  const long s0 = lv * 4 + 2 * q;  // the left-biased system; s0 + 1 the right-biased one
  if (C.R.crweno) {
    bool zp = false;
    for (int j = 0; j < 2; j++) {
      const long o = (s0 + j) * (N + 1);
      long_system(L + o, L + f + o, L + 2 * f + o, L + 3 * f + o, N, red, carry, C.R.plain_start != 0, zp);
    }
    if (zp) atomicOr(C.status, 1);
  }
  // interface arrays: split mode uL, uR (q 0) or fL, fR (q 1); paired mode
  // 0.5*(uR - uL) or 0.5*(fL + fR)
  const Global<double> *io = dir ? C.iy : C.ix;
  const long line = ((long)v * S.nlines + l) * (N + 1);
  const double *xl = L + 3 * f + s0 * (N + 1), *xr = xl + (N + 1);
  for (int k = threadIdx.x; k <= N; k += kLongTeam) {
    if (C.paired) io[q][line + k] = q ? 0.5 * (xl[k] + xr[k]) : 0.5 * (xr[k] - xl[k]);
    else {
      io[2 * q][line + k] = xl[k];
      io[2 * q + 1][line + k] = xr[k];
    }
  }
}

// ---------------------------------------------------------------------------
// Upwinding.
//  NS2D Roe: NavierStokes2DUpwind.c:26-92 with navierstokes2d.h:115-311 --
//   |A| = R |D| L built as the 4x4 flow block (the species block of the
//   reference's dense n x n product is diagonal: R = L = I, D = vn), Harten
//   entropy fix delta = 1e-6.
//  Euler1D Roe: Euler1DUpwind.c:27-93 (no entropy fix); rf-char :107-190.
// ---------------------------------------------------------------------------
// An interface: offset of its variable 0 in the interface arrays and of the cells
// beside it in the state, and how far apart variables are in each.
struct Iface {
  long ii, vs, cL, cR, pl;
};
// In paired mode io[0] holds 0.5*(uR - uL) and io[1] 0.5*(fL + fR) (the only
// combinations the Roe flux uses); in split mode io[0..3] hold uL uR fL fR.
#define UD(m) (PAIR ? io[0][(m) * a.vs + a.ii] : 0.5 * (io[1][(m) * a.vs + a.ii] - io[0][(m) * a.vs + a.ii]))
#define FS(m) (PAIR ? io[1][(m) * a.vs + a.ii] : 0.5 * (io[2][(m) * a.vs + a.ii] + io[3][(m) * a.vs + a.ii]))

template <int DIR, int PAIR, class IO>
__device__ __forceinline__ void upwind_ns2d_roe(const Iface &a, int nv, double g, const double *__restrict__ q, const IO *io,
                                                double *__restrict__ fI, bool species) {
  const double uLc[4] = {q[a.cL], q[a.pl + a.cL], q[2 * a.pl + a.cL], q[3 * a.pl + a.cL]};
  const double uRc[4] = {q[a.cR], q[a.pl + a.cR], q[2 * a.pl + a.cR], q[3 * a.pl + a.cR]};
  double ud[4], fs[4], fo[4];
#pragma unroll
  for (int m = 0; m < 4; m++) {
    ud[m] = UD(m);
    fs[m] = FS(m);
  }
  const double Dsp = roe_ns2d<DIR>(g, uLc, uRc, ud, fs, fo);
#pragma unroll
  for (int m = 0; m < 4; m++) fI[m * a.vs + a.ii] = fo[m];
  if (species)  // else the reconstruction has written them
    for (int m = 4; m < nv; m++) fI[m * a.vs + a.ii] = FS(m) - Dsp * UD(m);
}

template <int PAIR, class IO>
__device__ __forceinline__ void upwind_e1d(const Iface &a, int nv, double g, int mode, const double *__restrict__ q, const IO *io,
                                           double *__restrict__ fI) {
  const double uLc[3] = {q[a.cL], q[a.pl + a.cL], q[2 * a.pl + a.cL]};
  const double uRc[3] = {q[a.cR], q[a.pl + a.cR], q[2 * a.pl + a.cR]};
  const long vs = a.vs, ii = a.ii;
  if (mode == 0 || mode == 3) {
    double ud[3], fs[3], fo[3];
    for (int m = 0; m < 3; m++) {
      ud[m] = UD(m);
      fs[m] = FS(m);
    }
    const double c = mode == 3 ? rusanov_e1d(g, uLc, uRc) : roe_e1d(g, uLc, uRc, ud, fs, fo);
    for (int m = 0; m < 3; m++) fI[m * vs + ii] = mode == 3 ? fs[m] - c * ud[m] : fo[m];
    for (int m = 3; m < nv; m++) fI[m * vs + ii] = FS(m) - c * UD(m);
    return;
  }
  const double *uL = io[0] + ii, *uR = io[1] + ii, *fL = io[2] + ii, *fR = io[3] + ii;
  double b[4][3], fo[3], es[3];
  for (int m = 0; m < 3; m++) {
    b[0][m] = uL[m * vs];
    b[1][m] = uR[m * vs];
    b[2][m] = fL[m * vs];
    b[3][m] = fR[m * vs];
  }
  rf_e1d(g, mode == 2, uLc, uRc, b[0], b[1], b[2], b[3], fo, es);
  for (int m = 0; m < 3; m++) fI[m * vs + ii] = fo[m];
  for (int m = 3; m < nv; m++)
    fI[m * vs + ii] = rf_pick(es[0], es[1], es[2], uL[m * vs], uR[m * vs], fL[m * vs], fR[m * vs], mode == 2);
}

// Split mode only: uL, uR, fL, fR in io[0..3].
template <int DIR, class IO>
__device__ __forceinline__ void upwind_ns2d_rf(const Iface &a, int nv, double g, bool llf, const IO *io,
                                               double *__restrict__ fI) {
  const long vs = a.vs, ii = a.ii;
  const double *uL = io[0] + ii, *uR = io[1] + ii, *fL = io[2] + ii, *fR = io[3] + ii;
  const double uLk[4] = {uL[0], uL[vs], uL[2 * vs], uL[3 * vs]};
  const double uRk[4] = {uR[0], uR[vs], uR[2 * vs], uR[3 * vs]};
  const double fLk[4] = {fL[0], fL[vs], fL[2 * vs], fL[3 * vs]};
  const double fRk[4] = {fR[0], fR[vs], fR[2 * vs], fR[3 * vs]};
  double fo[4], es[3];
  rf_ns2d<DIR>(g, llf, uLk, uRk, fLk, fRk, fo, es);
#pragma unroll
  for (int i = 0; i < 4; i++) fI[i * vs + ii] = fo[i];
  for (int m = 4; m < nv; m++)
    fI[m * vs + ii] = rf_pick(es[0], es[1], es[2], uL[m * vs], uR[m * vs], fL[m * vs], fR[m * vs], llf);
}

template <int DIR, int PAIR, class IO>
__device__ __forceinline__ void upwind_ns2d_rusanov(const Iface &a, int nv, double g, const double *__restrict__ q,
                                                    const IO *io, double *__restrict__ fI) {
  const double uLc[4] = {q[a.cL], q[a.pl + a.cL], q[2 * a.pl + a.cL], q[3 * a.pl + a.cL]};
  const double uRc[4] = {q[a.cR], q[a.pl + a.cR], q[2 * a.pl + a.cR], q[3 * a.pl + a.cR]};
  const double alpha = rusanov_ns2d<DIR>(g, uLc, uRc);
  for (int m = 0; m < nv; m++) fI[m * a.vs + a.ii] = FS(m) - alpha * UD(m);
}

#undef UD
#undef FS

__global__ void __launch_bounds__(256) k_upwind(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage >= C.nstages) return;
  const long nX = (long)(C.Sx.N + 1) * C.Sx.nlines;
  const long nY = (C.G.ndims == 2) ? (long)(C.Sy.N + 1) * C.Sy.nlines : 0;
  if (t >= nX + nY) return;
  auto at = [&](const SweepGeom &S, long it) {
    const int k = (int)(it % (S.N + 1)), l = (int)(it / (S.N + 1));
    const long c = S.base + (long)l * S.line_stride + k;
    return Iface{it, (long)S.nlines * (S.N + 1), c - 1, c, S.plane};
  };
  const int nv = C.G.nv, mode = C.upwind;
  const double g = C.P.gamma;
  if (C.model == 1) {
    if (C.paired) upwind_e1d<1>(at(C.Sx, t), nv, g, mode, C.U, C.ix, C.fIx);
    else upwind_e1d<0>(at(C.Sx, t), nv, g, mode, C.U, C.ix, C.fIx);
  } else if (mode == 1 || mode == 2) {  // rf-char, llf-char
    if (t < nX) upwind_ns2d_rf<0>(at(C.Sx, t), nv, g, mode == 2, C.ix, C.fIx);
    else upwind_ns2d_rf<1>(at(C.Sy, t - nX), nv, g, mode == 2, C.iy, C.fIy);
  } else if (mode == 3) {  // rusanov
    if (t < nX) {
      if (C.paired) upwind_ns2d_rusanov<0, 1>(at(C.Sx, t), nv, g, C.U, C.ix, C.fIx);
      else upwind_ns2d_rusanov<0, 0>(at(C.Sx, t), nv, g, C.U, C.ix, C.fIx);
    } else {
      if (C.paired) upwind_ns2d_rusanov<1, 1>(at(C.Sy, t - nX), nv, g, C.UT, C.iy, C.fIy);
      else upwind_ns2d_rusanov<1, 0>(at(C.Sy, t - nX), nv, g, C.UT, C.iy, C.fIy);
    }
  } else if (t < nX) {  // the species' fluxes may be the reconstruction's
    if (C.paired) upwind_ns2d_roe<0, 1>(at(C.Sx, t), nv, g, C.U, C.ix, C.fIx, !C.fuse_sp);
    else upwind_ns2d_roe<0, 0>(at(C.Sx, t), nv, g, C.U, C.ix, C.fIx, true);
  } else {
    if (C.paired) upwind_ns2d_roe<1, 1>(at(C.Sy, t - nX), nv, g, C.UT, C.iy, C.fIy, !C.fuse_sp);
    else upwind_ns2d_roe<1, 0>(at(C.Sy, t - nX), nv, g, C.UT, C.iy, C.fIy, true);
  }
}

// Upwind on the reference's layouts (a point's components contiguous), one thread
// per interface in memory order: a wave's threads take all of the cache lines
// they touch.  With the arrays changed to planes and back around k_upwind a call
// was seven launches of 6 to 20 us; 384 x 250, 11 variables, now one of 27.
__global__ void __launch_bounds__(256) k_dev_upwind(AosGrid A, int model, int mode, double g, int dir,
                                                    const double *uL, const double *uR, const double *fL,
                                                    const double *fR, const double *u, double *fI) {
  const int N = dir ? A.ny : A.nx, nl = A.ndims == 2 ? (dir ? A.nx : A.ny) : 1;
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= (long)(N + 1) * nl) return;
  const int k = (int)(dir ? p / A.nx : p % (N + 1)), l = (int)(dir ? p % A.nx : p / (N + 1));
  const long nxg = A.nx + 2 * A.g;
  const long row = A.ndims == 2 ? (dir ? k : l) + A.g : 0, cR = (row * nxg + (dir ? l : k) + A.g) * A.nv;
  const Iface a = {p * A.nv, 1, cR - (dir ? nxg : 1) * A.nv, cR, 1};
  const double *io[4] = {uL, uR, fL, fR};
  if (model == 1) upwind_e1d<0>(a, A.nv, g, mode, u, io, fI);
  else if (mode == 1 || mode == 2) dir ? upwind_ns2d_rf<1>(a, A.nv, g, mode == 2, io, fI) : upwind_ns2d_rf<0>(a, A.nv, g, mode == 2, io, fI);
  else if (mode == 3) dir ? upwind_ns2d_rusanov<1, 0>(a, A.nv, g, u, io, fI) : upwind_ns2d_rusanov<0, 0>(a, A.nv, g, u, io, fI);
  else dir ? upwind_ns2d_roe<1, 0>(a, A.nv, g, u, io, fI, true) : upwind_ns2d_roe<0, 0>(a, A.nv, g, u, io, fI, true);
}

// Conservation check, boundary part: the interface fluxes on the domain
// boundary summed over the lines in index order (HyperbolicFunction.c:104-110),
// one thread per variable; after the last stage the step's integral
// sum_s dt b_s (stage sums) (TimeRK.c:86-97), weighted by the face elements
// (BoundaryIntegral.c:37-58), is added to the case's total.
__global__ void __launch_bounds__(256) k_bflux(CASE_ARGS) {
  CASE_PREAMBLE
  if (stage >= C.nstages) return;
  const int nv = C.G.nv, nd = C.G.ndims;
  if (t >= nv) return;
  const int v = (int)t, nf = 2 * nd * nv;
  double *bf = C.bflux + (long)stage * nf;
  for (int d = 0; d < nd; d++) {
    const SweepGeom &S = d ? C.Sy : C.Sx;
    const double *fI = d ? C.fIy : C.fIx;
    const int N = S.N, nl = S.nlines;
    double lo = 0.0, hi = 0.0;
    for (int l = 0; l < nl; l++) {
      const long a = ((long)v * nl + l) * (N + 1);
      lo -= fI[a];
      hi += fI[a + N];
    }
    bf[(2 * d + 0) * nv + v] = lo;
    bf[(2 * d + 1) * nv + v] = hi;
  }
  if (stage != C.nstages - 1) return;
  double local = 0.0;
  for (int d = 0; d < nd; d++) {
    double step[2];
    for (int f = 0; f < 2; f++) {
      double sb = 0.0;
      for (int s = 0; s < C.nstages; s++) sb += (C.dt * C.b[s]) * C.bflux[(long)s * nf + (2 * d + f) * nv + v];
      step[f] = sb;
    }
    local += step[0] * C.dS[d];
    local += step[1] * C.dS[d];
  }
  C.tbi[v] += 1.0 * local;
}

// ---------------------------------------------------------------------------
// RHS assembly at interior points: rhs = -hyp + par + source
// (TimeRHSFunctionExplicit.c:55-74).  hyp = dxinv (fI[k+1] - fI[k]) summed
// over the dimensions in order (HyperbolicFunction.c:97-112): the x part from
// the x-sweep interfaces (contiguous along x), the y part from the y-sweep
// interfaces, which are contiguous along y and pass through an LDS tile;
// par: derivatives of the viscous fluxes; source: ChemistrySource
// (ChemistrySolve.c:18-115, chemistry.h:30-127) with the photon density of
// the Gaussian pulse at the stage time.
// ---------------------------------------------------------------------------
// component c (variable c + 1) of the parabolic term
// at point (i, j), byte offset o of the ghosted planes
__device__ __forceinline__ double viscous_par(const CaseDev &C, int c, int i, int j, size_t o) {
  const Grid &G = C.G;
  const PhysParams &P = C.P;
  const long pl = (long)G.nxg * G.nyg;
  const double dxi = C.dxinv[G.g + i], dyi = C.dxinv[(G.nx + 2 * G.g) + G.g + j];
  const double *Fx = C.FV + c * pl, *Fy = C.FV + (3 + c) * pl;
  const size_t row = 8 * (size_t)G.nxg;
  double dfx, dfy;
  if (P.par4) {
    const double t12 = 1.0 / 12.0;
    dfx = (elem(Fx, o - 16) - 8 * elem(Fx, o - 8) + 8 * elem(Fx, o + 8) - elem(Fx, o + 16)) * t12;
    dfy = (elem(Fy, o - 2 * row) - 8 * elem(Fy, o - row) + 8 * elem(Fy, o + row) - elem(Fy, o + 2 * row)) * t12;
  } else {
    dfx = 0.0 * elem(Fx, o + 8) - (-1.0) * elem(Fx, o) + (-1.0) * elem(Fx, o - 8);
    dfy = 0.0 * elem(Fy, o + row) - (-1.0) * elem(Fy, o) + (-1.0) * elem(Fy, o - row);
  }
  const double px = dxi * dfx;
  return px + dyi * dfy;
}

// Sponge zones act as a source (BCSponge.c:29-74, called by
// SourceFunction.c:44-58 after the physics source): zone by zone,
// s - sigma (U - uref) with sigma linear in the coordinate along the zone's dim.
__device__ __forceinline__ bool in_sponge(const CaseDev &C, int i, int j) {
  for (int z = 0; z < C.nzones; z++) {
    const Zone &Z = C.zones[z];
    if (Z.kind == Z_SPONGE && i >= Z.is[0] && i < Z.ie[0] && j >= Z.is[1] && j < Z.ie[1]) return true;
  }
  return false;
}

__device__ __forceinline__ double sponge(const CaseDev &C, int i, int j, int v, long p, double s) {
  const Grid &G = C.G;
  for (int z = 0; z < C.nzones; z++) {
    const Zone &Z = C.zones[z];
    if (Z.kind != Z_SPONGE || i < Z.is[0] || i >= Z.ie[0] || j < Z.is[1] || j >= Z.ie[1]) continue;
    const double x = Z.dim ? C.xc[(G.nx + 2 * G.g) + G.g + j] : C.xc[G.g + i];
    const double sigma = (Z.face > 0) ? (x - Z.xmin) / (Z.xmax - Z.xmin) : (x - Z.xmax) / (Z.xmin - Z.xmax);
    s -= (sigma * (C.U[(long)v * G.plane + p] - C.bcvals[Z.vals + v]));
  }
  return s;
}

// the Gaussian pulse at the stage time (ChemistrySolve.c:36-43); the photon
// density reaching layer 0 is its product with the beam map
__device__ __forceinline__ double chem_pulse(const CaseDev &C, int stage, double t0) {
  const PhysParams &P = C.P;
  const double time = t0 + C.c[stage] * C.dt;
  if (!(time > P.t_start_norm)) return 0.0;
  const double sigma = P.t_pulse_norm / 2.35482;
  const double tp = time - (P.t_start_norm + P.t_pulse_norm);
  return P.I0 * exp(-(tp * tp) / (2 * sigma * sigma));
}

// Photochemistry source of variable v (chemistry.h:30-127, ChemistrySolve.c:
// 45-110): a species' own term, or the energy's, which is the last layer's
// heating.  The other variables have none.  n(q): species q of the layer; nh:
// the photon density reaching it.
struct ChemVar {
  int layer, m;   // m: species of the layer, -1 the energy
  unsigned need;  // what the source reads, bits 0..6 the species of the layer, bit 7 the photons
};
__device__ __forceinline__ ChemVar chem_of(const PhysParams &P, int v) {
  ChemVar c = {P.nlayers - 1, -1, 0xFF};
  if (v >= P.nflow) {
    c.layer = P.nlayers > 1 ? (v - P.nflow) / P.z_stride : 0;
    c.m = v - P.nflow - P.z_stride * c.layer;
    c.need = c.m == 1 ? 0xBE : c.m == 2 ? 0xC7 : c.m == 3 ? 0x9A : c.m == 4 ? 0x16 : c.m == 5 ? 0x27 : 0;
  }
  return c;
}
template <class F>
__device__ __forceinline__ double chem_term(const PhysParams &P, int m, F n, double nh) {
  if (m < 0) {
    const double nO3 = n(1), nO2 = n(0), n1D = n(2), n1Dg = n(3), n3Su = n(4), n1Sg = n(5), nCO2 = n(6);
    return ((P.q0a * P.k0a + P.q0b * P.k0b) * nh * nO3 + (P.q1a * P.k1a + P.q1b * P.k1b) * nO2 * n1D +
            (P.q2a * P.k2a + P.q2b * P.k2b) * nO3 * n1D + (P.q3a * P.k3a + P.q3b * P.k3b) * nO3 * n1Sg +
            P.q4 * P.k4 * n1D * nCO2 + P.q5 * P.k5 * nO3 * n3Su + P.q6 * P.k6 * n1Dg * nO3) /
           P.ch_gm1;
  }
  switch (m) {
    case 1: {
      const double nO3 = n(1);
      return -(P.k0a + P.k0b) * nh * nO3 - (P.k2a + P.k2b) * nO3 * n(2) - (P.k3a + P.k3b) * nO3 * n(5) -
             P.k5 * nO3 * n(4) - P.k6 * n(3) * nO3;
    }
    case 2: {
      const double nO3 = n(1), n1D = n(2);
      return P.k0a * nh * nO3 - (P.k1a + P.k1b) * n1D * n(0) - (P.k2a + P.k2b) * n1D * nO3 - P.k4 * n1D * n(6);
    }
    case 3: return P.k0a * nh * n(1) + P.k5 * n(1) * n(4) - P.k6 * n(3) * n(1);
    case 4: return P.k2a * n(1) * n(2) - P.k5 * n(1) * n(4);
    case 5: return P.k1a * n(2) * n(0) - (P.k3a + P.k3b) * n(1) * n(5);
    default: return 0.0;
  }
}
// photon density reaching layer iz at byte offset o, from the pulse at the stage
// time (chem_pulse) and the beam map
__device__ __forceinline__ double chem_photons(const CaseDev &C, int iz, size_t o, double hs, double imap) {
  const PhysParams &P = C.P;
  double nh = (hs * imap) / P.hnu_den;
  for (int z = 0; z < iz; z++)
    nh = nh * (1.0 - P.damp_coef * elem(C.U + (long)(P.nflow + P.z_stride * z + 1) * C.G.plane, o));
  return nh;
}
// the species of a layer
__device__ __forceinline__ const double *chem_planes(const CaseDev &C, int layer) {
  return C.U + (long)(C.P.nflow + C.P.z_stride * layer) * C.G.plane;
}

// rhs of variable v at interior point (i, j), ghosted offset p, with its
// source added (SourceFunction.c:21-60): chemistry, then the sponge zones
__device__ __forceinline__ double with_source(const CaseDev &C, int v, int i, int j, long p, double hs, double r) {
  const bool chem = C.P.chem && v >= C.P.nflow - 1;
  double s = 0.0;
  if (chem) {
    const size_t o = 8 * (size_t)p;
    const ChemVar cv = chem_of(C.P, v);
    const double *n = chem_planes(C, cv.layer);
    const double nh = cv.need >> 7 ? chem_photons(C, cv.layer, o, hs, elem(C.imap, o)) : 0.0;
    s = chem_term(C.P, cv.m, [&](int q) { return elem(n + q * C.G.plane, o); }, nh);
  }
  if (C.sponge && in_sponge(C, i, j)) return r + sponge(C, i, j, v, p, s);
  return chem ? r + s : r;
}

// One variable of one 32 x 32 tile per block, a row of tiles variable by variable
// in neighbouring blocks of one XCD.  Bound by memory latency on small grids and
// by HBM on large ones.  A block has one exchange through LDS (the y-sweep
// interfaces, which are contiguous along y) and no serial walk over the variables:
// a tile's latency is paid once, not once per variable, a grid of few tiles has
// nv times as many blocks, and the source is added before the one store of a
// value.  Every load, the species of the source among them, is issued before the
// first is needed; the pulse is formed by one wave.  512 threads with two points
// each: with four the kernel takes 152 registers and the grids of few tiles have
// half the waves (k_next, 128 x 97: 11.9 -> 9.2 us, 201 x 201: 6.4 -> 5.7; large
// grids alike, and so are they with 16, 20 or 24 waves a CU).  With a tile per
// block walking all variables k_assemble took, nv 11: 128 x 97 53.3 -> 10.5 us,
// 600 x 343 59.4 -> 26, 1024^2 119 -> 115, 2048 x 1531 368 -> 336 us.
constexpr int kTileThreads = 512;
struct Tile {
  double y[32][33];     // y-sweep interfaces
  double pulse;         // chem_pulse of the stage
  double next[32][33];  // the state k_next writes, for the transposed copy and the ghost points
};

// NEXT: the values of the next stage's state (or the new solution) follow from
// the right-hand side at once (k_next)
template <bool NEXT>
__device__ __forceinline__ void assemble_tile(const CaseDev &C, int stage, int block, int first, Tile &sh) {
  const Grid &G = C.G;
  const int nv = G.nv;
  constexpr int R = kTileThreads / 32, Q = 32 / R;  // rows of the tile at a time, and of a thread
  auto &tl = sh.y;
  const int ntx = (G.nx + 31) / 32;
  const int nb = ntx * ((G.ny + 31) / 32) * nv;  // the case's blocks are padded to a multiple of eight
  const int id = xcd_order(block, (nb + 7) & ~7, first);
  if (id >= nb) return;
  const int strip = (unsigned)id / (unsigned)ntx, row = (unsigned)strip / (unsigned)nv, v = strip - row * nv;
  const int i0 = (id - strip * ntx) * 32, j0 = row * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int i = i0 + tx;
  const long pl = (long)v * G.plane;
  // Points outside the grid read the nearest one inside and are not stored, so
  // that every load is issued without a branch (a branch would wait for the
  // loads before it).
  const int ic = min(i, G.nx - 1);
  auto jq = [&](int q) { return min(j0 + ty + R * q, G.ny - 1); };
  size_t o[Q];  // byte offset of the thread's points in a plane
#pragma unroll
  for (int q = 0; q < Q; q++) o[q] = 8 * ((size_t)(jq(q) + G.gy) * G.nxg + (ic + G.g));
  // y-sweep interfaces of lines i0..i0+31, interfaces j0..j0+32
  const double *fIx = C.fIx + (long)v * G.ny * (G.nx + 1), *fIy = C.fIy + (long)v * G.nx * (G.ny + 1);
  double fy[Q], fy32 = 0.0;
#pragma unroll
  for (int q = 0; q < Q; q++)
    fy[q] = elem(fIy, 8 * ((size_t)min(i0 + ty + R * q, G.nx - 1) * (G.ny + 1) + min(j0 + tx, G.ny)));
  // interface j0 + 32 of line i0 + the thread's index, by the first 32 threads
  if (threadIdx.x < 32) fy32 = elem(fIy, 8 * ((size_t)ic * (G.ny + 1) + min(j0 + 32, G.ny)));
  const bool visc = C.P.viscous && (C.terms & 2) && v >= 1 && v <= 3;
  double hx[Q], add[Q];
  {
    double x0[Q], x1[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const size_t a = 8 * ((size_t)jq(q) * (G.nx + 1) + ic);
      x0[q] = elem(fIx, a);
      x1[q] = elem(fIx, a + 8);
    }
    const double dxi = C.dxinv[G.g + ic];
#pragma unroll
    for (int q = 0; q < Q; q++) hx[q] = dxi * (x1[q] - x0[q]);
  }
  // the solution and the stages before, with their coefficients in what follows
  const int ns = C.nstages;
  const bool last = stage == ns - 1;
  double un[Q], prev[3][Q], cf[4];
  if (NEXT) {
#pragma unroll
    for (int q = 0; q < Q; q++) un[q] = elem(C.u + pl, o[q]);
#pragma unroll
    for (int j = 0; j < 4; j++) cf[j] = j <= stage ? C.dt * (last ? C.b[j] : C.A[(stage + 1) * ns + j]) : 0.0;
#pragma unroll
    for (int j = 0; j < 3; j++)
      if (j < stage && (last || cf[j] != 0.0))
#pragma unroll
        for (int q = 0; q < Q; q++) prev[j][q] = elem(C.Udot[j] + pl, o[q]);
  }
#pragma unroll
  for (int q = 0; q < Q; q++) add[q] = visc ? viscous_par(C, v - 1, ic, jq(q), o[q]) : 0.0;
  // what the variable's source reads
  const bool chem = C.P.chem && (C.terms & 4) && v >= C.P.nflow - 1;
  const ChemVar cv = chem ? chem_of(C.P, v) : ChemVar{0, 0, 0};
  const unsigned need = cv.need;
  const double *species = chem_planes(C, cv.layer);
  double sp[8][Q];
#pragma unroll
  for (int k = 0; k < 7; k++)
    if (need >> k & 1)
#pragma unroll
      for (int q = 0; q < Q; q++) sp[k][q] = elem(species + k * G.plane, o[q]);
  if (need >> 7)
#pragma unroll
    for (int q = 0; q < Q; q++) sp[7][q] = elem(C.imap, o[q]);
  const double t0 = C.time[NEXT && stage ? 1 : 0];
  if (NEXT && block == 0 && threadIdx.x == 0) {  // the blocks read the other of the two
    if (stage == 0) C.time[1] = t0;
    else if (last) C.time[0] = t0 + C.dt;
  }
#pragma unroll
  for (int q = 0; q < Q; q++) tl[ty + R * q][tx] = fy[q];
  if (threadIdx.x < 32) tl[threadIdx.x][32] = fy32;
  if (need >> 7 && threadIdx.x < 64) sh.pulse = chem_pulse(C, stage, t0);
  lds_barrier();
  double sv[Q] = {};
  if (need) {
    const double hs = sh.pulse;
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const double nh = need >> 7 ? chem_photons(C, cv.layer, o[q], hs, sp[7][q]) : 0.0;
      sv[q] = chem_term(C.P, cv.m, [&](int k) { return sp[k][q]; }, nh);
    }
  }
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int jl = ty + R * q, j = j0 + jl;
    const double hyp = hx[q] + C.dxinv[(G.nx + 2 * G.g) + G.g + jq(q)] * (tl[tx][jl + 1] - tl[tx][jl]);
    double r = (C.terms & 1) ? -hyp : 0.0;
    if (visc) r = r + add[q];
    if (i < G.nx && j < G.ny) {
      // chemistry, then the sponge zones (SourceFunction.c:21-60)
      if (C.sponge && (C.terms & 4) && in_sponge(C, i, j)) r = r + sponge(C, i, j, v, o[q] / 8, sv[q]);
      else if (chem) r = r + sv[q];
      if (!NEXT || !last) elem(C.Udot[stage] + pl, o[q]) = r;
      if (NEXT) {
        double x = un[q];
#pragma unroll
        for (int m = 0; m < 3; m++)
          if (m < stage && (last || cf[m] != 0.0)) x += cf[m] * prev[m][q];
        if (last || cf[stage] != 0.0) x += cf[stage] * r;
        if (last) elem(C.u + pl, o[q]) = x;
        elem(C.Un + pl, o[q]) = x;
        sh.next[jl][tx] = x;
      }
    }
  }
  if (!NEXT) return;
  lds_barrier();
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int il = ty + R * q;
    if (i0 + il < G.nx && j0 + tx < G.ny)
      elem(C.UT + pl, 8 * ((size_t)(i0 + il + G.g) * G.nyg + (j0 + tx + G.gy))) = sh.next[tx][il];
  }
  // ghost points whose source lies in the tile, of the faces that copy
  if (!C.push[0] || (i0 >= G.g && i0 + 32 <= G.nx - G.g && j0 >= G.g && j0 + 32 <= G.ny - G.g)) return;
#pragma unroll
  for (int f = 0; f < 4; f++) {
    const int kind = C.push[f], d = f >> 1, hi = f & 1;
    const int N = d ? G.ny : G.nx, No = d ? G.nx : G.ny, b0 = d ? j0 : i0, o0 = d ? i0 : j0;
    for (int e = threadIdx.x; e < 32 * G.g; e += kTileThreads) {
      const int m = e >> 5, o = e & 31, k = hi ? N + m : -1 - m;  // ghost position m along d
      const int src = (kind == 1 ? (hi ? m : N - 1 - m) : (hi ? N - 1 - m : m)) - b0;
      if (src < 0 || src >= 32 || o0 + o >= No) continue;
      const double x = d ? sh.next[src][o] : sh.next[o][src];
      const int gi = d ? o0 + o : k, gj = d ? k : o0 + o;
      C.Un[pl + (long)(gj + G.gy) * G.nxg + (gi + G.g)] = x;
      C.UT[pl + (long)(gi + G.g) * G.nyg + (gj + G.gy)] = x;
    }
  }
}

__global__ void __launch_bounds__(kTileThreads) k_assemble(CASE_ARGS) {
  CASE_PREAMBLE
  const int s = stage & 0xFF;
  if (s >= C.nstages || skipped(C, stage)) return;
  const Grid &G = C.G;
  if (G.ndims == 1) {
    const bool src = (C.P.chem || C.sponge) && (C.terms & 4);
    if (t >= (long)G.nx * G.nv) return;
    const int v = (int)(t / G.nx), i = (int)(t % G.nx);
    const long p = i + G.g;
    const long a = (long)v * (G.nx + 1) + i;
    const double hyp = C.dxinv[G.g + i] * (C.fIx[a + 1] - C.fIx[a]);
    double r = (C.terms & 1) ? -hyp : 0.0;
    if (src) r = with_source(C, v, i, 0, p, C.P.chem ? chem_pulse(C, s, *C.time) : 0.0, r);
    C.Udot[s][(long)v * G.plane + p] = r;
    return;
  }
  __shared__ Tile sh;
  assemble_tile<false>(C, s, (int)blockIdx.x - first, first, sh);
}

// The assembly with what follows from it point by point: the next stage's state
// (TimeRK.c:46-57, as stage_value) in both layouts, after the last stage the new
// solution (:86-99) and with it the next step's first state, and the ghost points
// that are copies of interior ones.  With k_stage and k_update apart a step had
// five launches more and 33 passes over a state's values, now 27.  Per stage, their
// share of k_update included: 128 x 97 17.4 -> 7.9 us, 201 x 201 12.0 -> 5.7,
// 600 x 343 46.8 -> 35.7, 1024^2 208 -> 193, 2048 x 1531 629 -> 622.
__global__ void __launch_bounds__(kTileThreads) k_next(CASE_ARGS) {
  CASE_PREAMBLE
  (void)t;
  if (stage >= C.nstages) return;
  __shared__ Tile sh;
  assemble_tile<true>(C, stage, (int)blockIdx.x - first, first, sh);
}

// u += (dt*b_s) * Udot_s stage by stage (TimeRK.c:86-99) at interior points;
// time += dt (TimePostStep.c:33).
__global__ void __launch_bounds__(256) k_update(CASE_ARGS) {
  CASE_PREAMBLE
  const Grid &G = C.G;
  const long nint = (long)G.nx * G.ny;
  if (skipped(C, stage) || t >= nint * G.nv) return;
  if (t == 0) *C.time = *C.time + C.dt;
  const int v = (int)(t / nint);
  const long q = t % nint;
  const int i = (int)(q % G.nx), j = (int)(q / G.nx);
  const long p = (long)v * G.plane + (long)(j + G.gy) * G.nxg + (i + G.g);
  double x = C.u[p];
  for (int s = 0; s < C.nstages; s++) x += (C.dt * C.b[s]) * C.Udot[s][p];
  C.u[p] = x;
}


// Per-block partial max CFL (Euler1DComputeCFL.c / NavierStokes2DComputeCFL.c)
// and sum of squared step differences (TimePostStep.c:41-53).
__global__ void __launch_bounds__(TB) k_cfl_norm(Grid G, int model, double gam, double dt,
                                                 const double *__restrict__ u, const double *__restrict__ u_prev,
                                                 const double *__restrict__ dxinv, double *__restrict__ partials) {
  __shared__ double smax[TB], ssum[TB];
  const long nint = (long)G.nx * G.ny;
  double mx = 0.0, sm = 0.0;
  for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < nint; t += (long)gridDim.x * blockDim.x) {
    const int i = (int)(t % G.nx), j = (int)(t / G.nx);
    const long p = (long)(j + G.gy) * G.nxg + (i + G.g);
    if (model == 1) {
      const double rho = u_prev[p], v = u_prev[G.plane + p] / rho;
      const double P = (u_prev[2 * G.plane + p] - 0.5 * rho * v * v) * (gam - 1.0);
      const double c = sqrt(gam * P / rho);
      const double l = (fabs(v) + c) * dt * dxinv[G.g + i];
      mx = l > mx ? l : mx;
    } else {
      const double rho = u_prev[p];
      const double vx = (rho == 0) ? 0 : u_prev[G.plane + p] / rho, vy = (rho == 0) ? 0 : u_prev[2 * G.plane + p] / rho;
      const double vsq = (vx * vx) + (vy * vy);
      const double P = (u_prev[3 * G.plane + p] - 0.5 * rho * vsq) * (gam - 1.0);
      const double c = sqrt(gam * P / rho);
      const double lx = (fabs(vx) + c) * dt * dxinv[G.g + i];
      const double ly = (fabs(vy) + c) * dt * dxinv[(G.nx + 2 * G.g) + G.g + j];
      mx = lx > mx ? lx : mx;
      mx = ly > mx ? ly : mx;
    }
    for (int v = 0; v < G.nv; v++) {
      const double d = u_prev[(long)v * G.plane + p] - u[(long)v * G.plane + p];
      sm += d * d;
    }
  }
  smax[threadIdx.x] = mx;
  ssum[threadIdx.x] = sm;
  __syncthreads();
  for (int s = TB / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      smax[threadIdx.x] = smax[threadIdx.x] > smax[threadIdx.x + s] ? smax[threadIdx.x] : smax[threadIdx.x + s];
      ssum[threadIdx.x] += ssum[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = smax[0];
    partials[2 * blockIdx.x + 1] = ssum[0];
  }
}


// Batched tridiagonal solve for the unit-level entry point, one team per
// system (tridiagLU.c:86-277 semantics with a_0 = c_{n-1} = 0, as in the
// reference's serial use): systems stored [n][ns], rows distributed over the
// team's lanes as in the reconstruction.
__global__ void __launch_bounds__(TB) k_tridiag(const double *__restrict__ a, const double *__restrict__ b,
                                                const double *__restrict__ c, double *__restrict__ x, int n, int ns,
                                                int T, int m, int *__restrict__ flag) {
  __shared__ double red[16];
  const int lane = threadIdx.x & (T - 1);
  const long d = (long)blockIdx.x * (TB / T) + threadIdx.x / T;
  const bool active = d < ns;
  const int lo = lane * m;
  int nr = n - lo;
  nr = nr < 0 ? 0 : (nr > m ? m : nr);
  if (!active) nr = 0;
  double A[kMaxRows], B[kMaxRows], Cc[kMaxRows], X[kMaxRows];
#pragma unroll
  for (int i = 0; i < kMaxRows; i++) {
    if (i < nr) {
      const long q = (long)(lo + i) * ns + d;
      A[i] = (lo + i == 0) ? 0.0 : a[q];
      B[i] = b[q];
      Cc[i] = (lo + i == n - 1) ? 0.0 : c[q];
      X[i] = x[q];
    } else {
      A[i] = 0.0; B[i] = 1.0; Cc[i] = 0.0; X[i] = 0.0;
    }
  }
  team_solve<kMaxRows>(A, B, Cc, X, nr, lane, T, lane == (n - 1) / m, 0.0, 0.0, red, flag, false);
#pragma unroll
  for (int i = 0; i < kMaxRows; i++)
    if (i < nr) x[(long)(lo + i) * ns + d] = X[i];
}

// The same for systems longer than one team covers: one thread per system,
// the sequential sweep itself (tridiagLU.c:133-150 and :243-255, a_0 = c_{n-1}
// = 0).  b receives the pivots b', x receives x' and then the solution.
__global__ void __launch_bounds__(TB) k_tridiag_seq(const double *__restrict__ a, double *b,
                                                    const double *__restrict__ c, double *__restrict__ x, int n,
                                                    int ns, int *__restrict__ flag) {
  const long d = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= ns) return;
  double bp = b[d], xp = x[d], cp = (n > 1) ? c[d] : 0.0;
  bool zp = bp == 0.0;
  for (int i = 1; i < n; i++) {
    const long q = (long)i * ns + d;
    const double fac = a[q] / bp;
    bp = b[q] - fac * cp;
    xp = x[q] - fac * xp;
    cp = (i == n - 1) ? 0.0 : c[q];
    zp = zp || bp == 0.0;
    b[q] = bp;
    x[q] = xp;
  }
  if (zp) atomicOr(flag, 1);
  double xn = x[(long)(n - 1) * ns + d] / b[(long)(n - 1) * ns + d];
  x[(long)(n - 1) * ns + d] = xn;
  for (int i = n - 2; i >= 0; i--) {
    const long q = (long)i * ns + d;
    xn = (x[q] - c[q] * xn) / b[q];
    x[q] = xn;
  }
}

__global__ void __launch_bounds__(TB) k_weno_weights(int kind, double c1, double c2, double c3,
                                                     const double *__restrict__ st, int count, double eps,
                                                     double *__restrict__ w) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const double *s = st + 5 * (long)t;
  double w1, w2, w3;
  weno_w_rt(kind, c1, c2, c3, s[0], s[1], s[2], s[3], s[4], eps, w1, w2, w3);
  w[3 * (long)t] = w1;
  w[3 * (long)t + 1] = w2;
  w[3 * (long)t + 2] = w3;
}

// ---------------------------------------------------------------------------
// Device-buffer operators on the reference's own array layouts, for callers
// that keep the reference's data structures on the device.  Ghosted arrays:
// every grid point with its ghost layers, x fastest, the nvars components of
// a point contiguous (include/hypar.h:106-111).  Interface arrays of
// dimension dir: the points of the grid with dim[dir]+1 interfaces along dir
// and no ghosts, same ordering (HyperbolicFunction.c:61-70).
// ---------------------------------------------------------------------------
// point offset of (i, j) (interior indices; ghosts negative) in a ghosted array
__device__ __forceinline__ long aos_point(const AosGrid &A, int i, int j) {
  return A.ndims == 2 ? (long)(j + A.g) * (A.nx + 2 * A.g) + (i + A.g) : (long)(i + A.g);
}
__device__ __forceinline__ long aos_points(const AosGrid &A) {
  return (long)(A.nx + 2 * A.g) * (A.ndims == 2 ? A.ny + 2 * A.g : 1);
}

// FluxFunction along dir at every point of the ghosted grid
__global__ void __launch_bounds__(TB) k_dev_flux(AosGrid A, int model, double gamma, int dir,
                                                 const double *__restrict__ u, double *__restrict__ f) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= aos_points(A)) return;
  const double *q = u + p * A.nv;
  double *o = f + p * A.nv;
  point_flux(model, dir, gamma, A.nv, [&](int m) { return q[m]; }, [&](int m, double x) { o[m] = x; });
}

// FirstDerivativePar along dir at every position (ghosts included) of every
// interior line across dir, one thread per (position, line, variable):
// FirstDerivativeFourthOrderCentral (FirstDerivativeFourthOrder.c:39-132) with
// par4, else FirstDerivativeFirstOrder (FirstDerivativeFirstOrder.c:20-95) with
// the given bias.  Points off the interior lines are left as they are.
__global__ void __launch_bounds__(TB) k_dev_fd(AosGrid A, int dir, int par4, int bias,
                                               const double *__restrict__ f, double *__restrict__ df) {
  const int N = dir ? A.ny : A.nx, g = A.g, nv = A.nv, P = N + 2 * g;
  const int nl = A.ndims == 2 ? (dir ? A.nx : A.ny) : 1;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)P * nl * nv) return;
  const int v = (int)(t % nv);
  const long r = t / nv;
  const int i = (int)(r % P) - g, l = (int)(r / P);
  auto F = [&](int k) { return f[aos_point(A, dir ? l : k, dir ? k : l) * nv + v]; };
  double d;
  if (par4) {
    const double t12 = 1.0 / 12.0;
    if (i == -g) d = (-25 * F(i) + 48 * F(i + 1) - 36 * F(i + 2) + 16 * F(i + 3) - 3 * F(i + 4)) * t12;
    else if (i == -g + 1) d = (-3 * F(i - 1) - 10 * F(i) + 18 * F(i + 1) - 6 * F(i + 2) + F(i + 3)) * t12;
    else if (i == N + g - 2) d = (-F(i - 3) + 6 * F(i - 2) - 18 * F(i - 1) + 10 * F(i) + 3 * F(i + 1)) * t12;
    else if (i == N + g - 1) d = (3 * F(i - 4) - 16 * F(i - 3) + 36 * F(i - 2) - 48 * F(i - 1) + 25 * F(i)) * t12;
    else d = (F(i - 2) - 8 * F(i - 1) + 8 * F(i + 1) - F(i + 2)) * t12;
  } else {
    const double mx = bias > 0 ? bias : 0, mn = bias < 0 ? bias : 0, bb = bias;
    if (i == -g) d = F(i + 1) - F(i);
    else if (i == N + g - 1) d = F(i) - F(i - 1);
    else d = mx * F(i + 1) - bb * F(i) + mn * F(i - 1);
  }
  df[aos_point(A, dir ? l : i, dir ? i : l) * nv + v] = d;
}

// SetInterpLimiterVar = WENOFifthOrderCalculateWeights{,Char}
// (WENOFifthOrderCalculateWeights.c:41-84, :112-237 and the M / Z / YC and
// characteristic variants): the nonlinear weights of every interface of dir
// on every interior line, for the left-biased flux, left-biased solution,
// right-biased flux and right-biased solution, in that order, set k at
// w + k*size.  Within a set, interface point p, variable v at p*nvars + v.
// Characteristic: the stencils are projected with the left eigenvectors of
// the Roe average of the two cells beside the interface (the flow block;
// species rows are the identity).  One thread per (interface, line).
template <int KIND>
__device__ __forceinline__ void dev_weights_at(const AosGrid &A, int model, double gam, int dir, int crweno,
                                               int characteristic, int no_limiting, double eps, int k, int l,
                                               const double *__restrict__ fC, const double *__restrict__ u,
                                               double *w1, double *w2, double *w3, long size) {
  const int nv = A.nv, N = dir ? A.ny : A.nx;
  const long p = dir ? (long)k * A.nx + l : (A.ndims == 2 ? (long)l * (A.nx + 1) + k : (long)k);
  auto at = [&](const double *a, int pos, int v) { return a[aos_point(A, dir ? l : pos, dir ? pos : l) * nv + v]; };
  double c1, c2, c3;
  if (crweno && k > 0 && k < N) { c1 = 0.2; c2 = 0.5; c3 = 0.3; }
  else { c1 = 0.1; c2 = 0.6; c3 = 0.3; }
  const int nf = characteristic ? (model == 1 ? 3 : 4) : 0;
  double L[4][4] = {{0}};
  if (nf == 3) {
    double a0, a1, a2;
    euler1d_roeavg(gam, at(u, k - 1, 0), at(u, k - 1, 1), at(u, k - 1, 2), at(u, k, 0), at(u, k, 1), at(u, k, 2),
                   a0, a1, a2);
    Eig3 E;
    euler1d_eig(gam, a0, a1, a2, E);
    for (int a = 0; a < 3; a++)
      for (int b = 0; b < 3; b++) L[a][b] = E.L[a][b];
  } else if (nf == 4) {
    const double uLc[4] = {at(u, k - 1, 0), at(u, k - 1, 1), at(u, k - 1, 2), at(u, k - 1, 3)};
    const double uRc[4] = {at(u, k, 0), at(u, k, 1), at(u, k, 2), at(u, k, 3)};
    double ua[4], R[4][4];
    ns2d_roeavg(gam, uLc, uRc, ua);
    if (dir) ns2d_eigvecs<1>(gam, ua, L, R);
    else ns2d_eigvecs<0>(gam, ua, L, R);
  }
  // stencil value of variable v at position pos (projected for the flow rows)
  auto sv = [&](const double *a, int pos, int v) {
    if (v >= nf) return at(a, pos, v);
    double y = L[v][0] * at(a, pos, 0);
    for (int b = 1; b < nf; b++) y = y + L[v][b] * at(a, pos, b);
    return y;
  };
  for (int set = 0; set < 4; set++) {  // LF, LU, RF, RU
    const double *a = (set & 1) ? u : fC;
    const bool left = set < 2;
    for (int v = 0; v < nv; v++) {
      double x1, x2, x3;
      if (no_limiting) {
        x1 = c1; x2 = c2; x3 = c3;
      } else if (left) {
        weno_w<KIND>(c1, c2, c3, sv(a, k - 3, v), sv(a, k - 2, v), sv(a, k - 1, v), sv(a, k, v), sv(a, k + 1, v),
                     eps, x1, x2, x3);
      } else {
        weno_w<KIND>(c1, c2, c3, sv(a, k + 2, v), sv(a, k + 1, v), sv(a, k, v), sv(a, k - 1, v), sv(a, k - 2, v),
                     eps, x1, x2, x3);
      }
      const long o = set * size + p * nv + v;
      w1[o] = x1;
      w2[o] = x2;
      w3[o] = x3;
    }
  }
}

__global__ void __launch_bounds__(TB) k_dev_weights(AosGrid A, int model, double gam, int dir, int kind,
                                                    int crweno, int characteristic, int no_limiting, double eps,
                                                    const double *__restrict__ fC, const double *__restrict__ u,
                                                    double *w1, double *w2, double *w3, long size) {
  const int N = dir ? A.ny : A.nx, nl = A.ndims == 2 ? (dir ? A.nx : A.ny) : 1;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)(N + 1) * nl) return;
  const int k = (int)(t % (N + 1)), l = (int)(t / (N + 1));
  switch (kind) {
    case 1: dev_weights_at<1>(A, model, gam, dir, crweno, characteristic, no_limiting, eps, k, l, fC, u, w1, w2, w3, size); break;
    case 2: dev_weights_at<2>(A, model, gam, dir, crweno, characteristic, no_limiting, eps, k, l, fC, u, w1, w2, w3, size); break;
    case 3: dev_weights_at<3>(A, model, gam, dir, crweno, characteristic, no_limiting, eps, k, l, fC, u, w1, w2, w3, size); break;
    default: dev_weights_at<0>(A, model, gam, dir, crweno, characteristic, no_limiting, eps, k, l, fC, u, w1, w2, w3, size); break;
  }
}

// Ghosted reference-layout array <-> the planar layouts of a case: the natural
// copy (x fastest) and, in 2D, the transposed copy (y fastest), either may be
// null.  One thread per (point, variable).  to_planar = 0 copies the other
// way, from the natural copy, at the ghost points only when ghosts_only.
__global__ void __launch_bounds__(TB) k_dev_planar(Grid G, const double *__restrict__ a, double *nat, double *tr,
                                                   int to_planar, int ghosts_only, double *out) {
  const long np = (long)G.nxg * G.nyg;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= np * G.nv) return;
  const int v = (int)(t % G.nv);
  const long p = t / G.nv;
  const int i = (int)(p % G.nxg) - G.g, j = (int)(p / G.nxg) - G.gy;
  const long pn = (long)v * G.plane + p;
  if (to_planar) {
    const double x = a[p * G.nv + v];
    if (nat) nat[pn] = x;
    if (tr) tr[(long)v * G.plane + (long)(i + G.g) * G.nyg + (j + G.gy)] = x;
    return;
  }
  const bool ghost = i < 0 || i >= G.nx || j < 0 || j >= G.ny;
  const bool corner = (i < 0 || i >= G.nx) && (j < 0 || j >= G.ny) && G.ndims == 2;
  if (ghosts_only && (!ghost || corner)) return;  // the reference never writes the corners
  out[p * G.nv + v] = nat[pn];
}

// Host states, point-major in pinned memory, to and from the planar layout
// (see transfer.hpp).  Bound by the host link, so consecutive lanes take
// consecutive values of the host side, and the planar side's short runs (the
// few points a wave covers of every variable) merge in L2.
__device__ __forceinline__ long pack_at(const Grid &G, long q0, unsigned e) {
  const unsigned v = e % (unsigned)G.nv;
  const long q = q0 + e / (unsigned)G.nv;
  const int i = (int)(q % G.nx), j = (int)(q / G.nx);
  return (long)v * G.plane + (long)(j + G.gy) * G.nxg + (i + G.g);
}
__global__ void __launch_bounds__(TB) k_pack(Grid G, const double *__restrict__ host, long q0, unsigned n,
                                             double *__restrict__ u) {
  const unsigned e = blockIdx.x * TB + threadIdx.x;
  if (e < n) u[pack_at(G, q0, e)] = host[e];
}
__global__ void __launch_bounds__(TB) k_unpack(Grid G, const double *__restrict__ u, long q0, unsigned n,
                                               double *__restrict__ host) {
  const unsigned e = blockIdx.x * TB + threadIdx.x;
  if (e < n) host[e] = u[pack_at(G, q0, e)];
}
__global__ void k_set_time(double *time, double t) { *time = t; }

// Interface arrays of one sweep: reference layout <-> line-major
// a[(v*nlines + l)*(N+1) + k].  One thread per (interface, line, variable).
__global__ void __launch_bounds__(TB) k_dev_iface(int ndims, int dir, int nx, int N, int nl, int nv,
                                                  const double *__restrict__ src, double *__restrict__ dst) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)(N + 1) * nl * nv) return;
  const int v = (int)(t % nv);
  const long r = t / nv;
  const int k = (int)(r % (N + 1)), l = (int)(r / (N + 1));
  const long p = dir ? (long)k * nx + l : (ndims == 2 ? (long)l * (N + 1) + k : (long)k);
  const long q = ((long)v * nl + l) * (N + 1) + k;
  dst[p * nv + v] = src[q];
}


}  // namespace

// ===========================================================================
// host side: work decomposition and launchers
// ===========================================================================

static const char *kKNames[K_NCLASS] = {"stage_bc", "ghost",  "flux",    "recon_ends",
                                        "recon_4",  "recon_6", "recon_8", "recon_10", "recon_12", "recon_14", "recon_16",
                                        "recon_w10", "recon_w12", "recon_w16", "long_rows", "long_solve",
                                        "cw_rows", "cw_solve", "weno", "upwind", "bflux",
                                        "assemble", "next", "ghost_next", "update", "flux_all",
                                        "line_4", "line_8", "tube", "tube_back"};
const char *kclass_name(int k) { return kKNames[k]; }

int cw_row_fields(int nflow, int nv) { return nflow * nflow + 16 * nv; }
int cw_back_fields(int nflow, int nv) { return 2 * nflow * nflow + nflow + 3 * (nv - nflow); }

bool team_shape(int N, int max_rows, int &team, int &rows) {
  if (max_rows < 1 || max_rows > kMaxRows) max_rows = kMaxRows;
  const int nrows = N - 1 > 1 ? N - 1 : 1;
  team = 1;
  while ((long)team * max_rows < nrows) team <<= 1;
  rows = (nrows + team - 1) / team;
  return team <= 256;
}

bool line_shape(int N, int rows, int &team) {
  team = 1;
  while ((long)team * rows < N - 1) team <<= 1;
  if (team > 256) return false;
  for (const ReconVariant &v : kRecon)
    if (v.rows == rows && v.wide == (team > 64)) return true;
  return false;
}

// A launch of a variant costs its latency once and its lanes' rows; the choice
// minimises the sum over the variants used, of all sets of variants.  Both terms
// are fitted to launches of nv 11 grids of side N (us; rows 4 6 8 10 12 14 16):
//   N  33: 14.4 16.7 17.2 19.1 21.0 22.2 23.9     N 257: 65.3 78.6 57.5 74.9 83.1 93.8 68.6
//   N 129: 28.8 32.7 25.7 27.9 31.1 33.7 36.4     N 385:   -   114  142  178  122  138  149
//   N 193: 51.8 42.7 48.7 57.5 46.9 51.9 53.5     N 513:   -    -   186  239  271  299  202
// (teams are powers of two, so a row count serves some lengths better than
// others; short segments have more waves to hide their chains, long ones less
// overhead per row).  Rows 16 only, the choice before, is the last column.
// Teams of 128 and 256 lanes (rows 10 12 16; - : more than 256 lanes):
//   N 1100: 1364 1406 1578     N 1281: 1596 1679 1872     N 1400: 3195 1852 2055     N 1537: 3531 2034 2311
//   N 1800: 4213 4370 2774     N 2049: 4852 5022 3141     N 2561: 6160 6452 7251     N 3073:   -  7837 8865
// and 10720 at 3600, 12420 at 4096, both 16 rows.  The fit gives 1631 at 1281 (10
// rows), 2087 at 1537 (12), 3276 at 2049 (16) and the fastest of each line above.
void choose_rows(const std::vector<SweepGeom *> &sweeps, const std::vector<int> &nvars) {
  static const double per_row[kNRecon] = {1.25, 1.10, 1.00, 1.06, 1.11, 1.10, 1.06, 1.44, 1.28, 1.13};
  auto latency = [](int v) { return 10.0 + 0.75 * kRecon[v].rows; };
  const int ns = (int)sweeps.size();
  for (int wide = 0; wide < 2; wide++) {  // lines of up to 64 * kMaxRows rows take narrow teams
    const int v0 = wide ? 7 : 0, n = wide ? kNRecon - 7 : 7;
    std::vector<int> idx;
    for (int s = 0; s < ns; s++)
      if ((sweeps[s]->N - 1 > 64 * kMaxRows) == (wide == 1)) idx.push_back(s);
    if (idx.empty()) continue;
    std::vector<double> work(idx.size() * n);
    std::vector<int> team(idx.size() * n);
    for (size_t k = 0; k < idx.size(); k++)
      for (int v = 0; v < n; v++) {
        const SweepGeom &S = *sweeps[idx[k]];
        const int rows = kRecon[v0 + v].rows;
        int T;
        const bool fits = line_shape(S.N, rows, T) && (T > 64) == kRecon[v0 + v].wide;
        team[k * n + v] = fits ? T : 0;
        work[k * n + v] = fits ? 1.57e-5 * per_row[v0 + v] * T * rows * (2.0 * S.nlines * nvars[idx[k]]) : 1e30;
      }
    auto total = [&](int set, std::vector<int> *pick) {
      double sum = 0.0;
      int used = 0;
      for (size_t k = 0; k < idx.size(); k++) {
        int best = -1;
        for (int v = 0; v < n; v++)
          if ((set >> v & 1) && (best < 0 || work[k * n + v] < work[k * n + best])) best = v;
        sum += work[k * n + best];
        used |= 1 << best;
        if (pick) (*pick)[k] = best;
      }
      for (int v = 0; v < n; v++)
        if (used >> v & 1) sum += latency(v0 + v);
      return sum;
    };
    int set = 1 << (n - 1);  // the longest segments fit every line
    double best = total(set, nullptr);
    for (int c = 1; c < 1 << n; c++) {
      const double t = total(c, nullptr);
      if (t < best) {
        best = t;
        set = c;
      }
    }
    std::vector<int> pick(idx.size());
    total(set, &pick);
    for (size_t k = 0; k < idx.size(); k++) {
      sweeps[idx[k]]->rows = kRecon[v0 + pick[k]].rows;
      sweeps[idx[k]]->team = team[k * n + pick[k]];
    }
  }
}

bool velocity_for_flux(const CaseDev &c) {
  return c.R.crweno && !c.R.characteristic && !c.unit && !c.Sx.longl && !c.Sy.longl &&
         c.G.nv > (c.model == 1 ? 3 : 4);
}

bool stage_tile_64(const CaseDev &c) { return c.G.ndims == 2 && (long)c.G.nx * c.G.ny >= 2048L * 2048L; }

bool species_in_recon(const CaseDev &c) {
  auto fits = [](const SweepGeom &S) { return !S.longl && (S.team == 32 || S.team == 64 || S.team == 128); };
  return c.G.ndims == 2 && c.model == 2 && c.paired && c.R.crweno && c.upwind == 0 && !c.R.characteristic &&
         c.G.nv > 4 && c.dsp[0] && c.dsp[1] && fits(c.Sx) && fits(c.Sy);
}

void case_blocks(const CaseDev &c, int blocks[K_NCLASS]) {
  const Grid &G = c.G;
  const bool two = (G.ndims == 2);
  auto nb = [](long n) { return (int)((n + TB - 1) / TB); };
  const int st = c.stage_tile == 64 ? 64 : 32;
  // the tile kernels' counts are padded to a multiple of eight, so that every
  // case's tiles start on one and can be taken in xcd_order
  auto pad8 = [](int n) { return (n + 7) & ~7; };
  blocks[K_GHOST] = nb(ghost_points(G) * G.nv);
  blocks[K_STAGE] = stage_blocks(G, st) + blocks[K_GHOST];
  auto faces = [&](long per) {  // blocks of `per` interfaces, the sweeps apart
    const long x = (long)(c.Sx.N + 1) * c.Sx.nlines, y = two ? (long)(c.Sy.N + 1) * c.Sy.nlines : 0;
    return (int)((x + per - 1) / per + (y + per - 1) / per);
  };
  const int nf = c.model == 1 ? 3 : 4;
  const bool weno = !c.R.crweno && !c.unit;
  blocks[K_FLUXALL] = nb(flux_items(c));
  blocks[K_ENDS] = nb(end_items(c));
  blocks[K_FLUX] = weno ? 0 : viscous_blocks(c) + blocks[K_ENDS] + blocks[K_FLUXALL];
  blocks[K_WENO] = weno ? viscous_blocks(c) + faces(kWenoTile) : 0;
  blocks[K_CWROWS] = blocks[K_CWSOLVE] = blocks[K_LROWS] = blocks[K_LSOLVE] = 0;
  for (int v = 0; v < kNRecon; v++) blocks[K_RECON + v] = 0;
  if (c.R.crweno && c.R.characteristic) {
    blocks[K_CWROWS] = nb((long)(c.Sx.N + 1) * c.Sx.nlines + (two ? (long)(c.Sy.N + 1) * c.Sy.nlines : 0));
    blocks[K_CWSOLVE] = nb(cw_x_span(c, nf) + (two ? cw_items(c.Sy, G.nv, nf) : 0));
  } else if (c.R.crweno) {
    for (int v = 0; v < kNRecon; v++) {
      if (recon_in(c.Sx, kRecon[v].rows, kRecon[v].wide)) blocks[K_RECON + v] += recon_sweep_blocks(c.Sx, G.nv);
      if (two && recon_in(c.Sy, kRecon[v].rows, kRecon[v].wide)) blocks[K_RECON + v] += recon_sweep_blocks(c.Sy, G.nv);
    }
    blocks[K_LROWS] = nb(long_rows(c.Sx, G.nv) + (two ? long_rows(c.Sy, G.nv) : 0));
    blocks[K_LSOLVE] = (int)(long_pairs(c.Sx, G.nv) + (two ? long_pairs(c.Sy, G.nv) : 0));  // a block per pair
  }
  blocks[K_UPWIND] = weno ? 0 : nb((long)(c.Sx.N + 1) * c.Sx.nlines + (two ? (long)(c.Sy.N + 1) * c.Sy.nlines : 0));
  blocks[K_BFLUX] = c.cons ? 1 : 0;
  blocks[K_ASSEMBLE] = pad8(two ? ((G.nx + 31) / 32) * ((G.ny + 31) / 32) * G.nv
                                 : (int)(((long)G.nx * G.nv + kTileThreads - 1) / kTileThreads));
  blocks[K_NEXT] = c.fused ? blocks[K_ASSEMBLE] : 0;
  blocks[K_GHOSTNEXT] = c.fused && !c.push[0] ? blocks[K_GHOST] : 0;
  blocks[K_UPDATE] = nb((long)G.nx * G.ny * G.nv);
  const int line = line_class(c);
  blocks[K_LINE4] = line == K_LINE4;
  blocks[K_LINE8] = line == K_LINE8;
  blocks[K_TUBE] = line == K_TUBE ? (G.nx + tube_core(c.nstages) - 1) / tube_core(c.nstages) : 0;
  blocks[K_TUBEBACK] = line == K_TUBE ? nb((long)G.nx * G.nv) : 0;
}

static KernFn class_kernel(const Plan &pl, int cls) {
  static const KernFn recon[] = {recon_kernel<4, false>(),  recon_kernel<6, false>(),  recon_kernel<8, false>(),
                                 recon_kernel<10, false>(), recon_kernel<12, false>(), recon_kernel<14, false>(),
                                 recon_kernel<16, false>(), recon_kernel<10, true>(),  recon_kernel<12, true>(),
                                 recon_kernel<16, true>()};
  static_assert(sizeof recon / sizeof recon[0] == kNRecon, "a kernel per variant");
  if (cls >= K_RECON && cls < K_RECON + kNRecon) return recon[cls - K_RECON];
  switch (cls) {
    case K_STAGE: return pl.stage64 ? k_stage64 : k_stage;
    case K_GHOST: return k_ghost;
    case K_FLUX: return k_flux;
    case K_FLUXALL: return k_flux_all;
    case K_ENDS: return k_recon_ends;
    case K_LROWS: return k_lrows;
    case K_LSOLVE: return k_lsolve;
    case K_CWROWS: return k_cw_rows;
    case K_CWSOLVE: return k_cw_solve;
    case K_WENO: return weno_kernel();
    case K_UPWIND: return k_upwind;
    case K_BFLUX: return k_bflux;
    case K_ASSEMBLE: return k_assemble;
    case K_NEXT: return k_next;
    case K_GHOSTNEXT: return k_ghost_next;
    default: return k_update;
  }
}

static void run(int cls, const CaseDev *d, const Plan &pl, int s, hipStream_t st, MarkFn mark, void *ctx) {
  if (pl.nblocks[cls] <= 0) return;
  const bool recon = cls >= K_RECON && cls < K_RECON + kNRecon;
  const int threads = recon ? recon_threads(kRecon[cls - K_RECON].wide)
                            : (cls == K_ASSEMBLE || cls == K_NEXT) ? kTileThreads : TB;
  if (mark) mark(ctx, cls, true, st);
  hipLaunchKernelGGL(class_kernel(pl, cls), dim3(pl.nblocks[cls]), dim3(threads), 0, st, d, pl.blockcase[cls],
                     pl.firstblock[cls], s);
  if (mark) mark(ctx, cls, false, st);
}

void launch_stage(const CaseDev *d, const Plan &pl, int s, hipStream_t st, MarkFn mark, void *ctx, int last) {
  run(K_STAGE, d, pl, s, st, mark, ctx);
  if (last <= K_GHOST) return;
  if (last == K_FLUX) {
    run(K_FLUXALL, d, pl, s, st, mark, ctx);
    return;
  }
  run(K_FLUX, d, pl, s, st, mark, ctx);
  for (int cls = K_RECON; cls <= K_ASSEMBLE; cls++)
    if (cls <= last) run(cls, d, pl, s, st, mark, ctx);
}

void launch_begin(const CaseDev *d, const Plan &pl, hipStream_t st, MarkFn mark, void *ctx) {
  if (pl.nfused) run(K_STAGE, d, pl, 0, st, mark, ctx);
}

void launch_step_stage(const CaseDev *d, const Plan &pl, int s, hipStream_t st, MarkFn mark, void *ctx) {
  const bool rest = pl.nfused < pl.ncases;
  if (pl.nfused) d += (long)s * pl.ncases;
  if (rest) run(K_STAGE, d, pl, s | kUnfused, st, mark, ctx);
  run(K_FLUX, d, pl, s, st, mark, ctx);
  for (int cls = K_RECON; cls <= K_BFLUX; cls++) run(cls, d, pl, s, st, mark, ctx);
  if (rest) run(K_ASSEMBLE, d, pl, s | kUnfused, st, mark, ctx);
  run(K_NEXT, d, pl, s, st, mark, ctx);
  run(K_GHOSTNEXT, d, pl, s, st, mark, ctx);
}

void launch_update(const CaseDev *d, const Plan &pl, hipStream_t st, MarkFn mark, void *ctx) {
  if (pl.nfused < pl.ncases) run(K_UPDATE, d, pl, kUnfused, st, mark, ctx);
}

void choose_push(CaseDev &c) {
  const int n[2] = {c.G.nx, c.G.ny};
  for (int f = 0; f < 4; f++) {
    const int d = f >> 1, face = f & 1 ? -1 : 1, o = 1 - d;
    c.push[f] = 0;
    if (c.G.ndims != 2 || n[d] < c.G.g) continue;
    int z = c.nzones - 1;  // the last zone of the face decides, if it covers the face
    while (z >= 0 && (c.zones[z].kind == Z_SPONGE || c.zones[z].dim != d || c.zones[z].face != face)) z--;
    if (z < 0) continue;
    const Zone &Z = c.zones[z];
    if (Z.is[o] > 0 || Z.ie[o] < n[o]) continue;
    // (a periodic zone takes its source without its offset along the face)
    if (Z.kind == Z_PERIODIC && Z.is[o] == 0) c.push[f] = 1;
    if (Z.kind == Z_EXTRAPOLATE) c.push[f] = 2;
  }
  if (!(c.push[0] && c.push[1] && c.push[2] && c.push[3])) memset(c.push, 0, sizeof c.push);
}

int cfl_norm_blocks(const Grid &G) {
  const long n = (long)G.nx * G.ny;
  long b = (n + TB - 1) / TB;
  return (int)(b < 1024 ? b : 1024);
}

void launch_cfl_norm(const Grid &G, int model, double gamma, double dt, const double *u, const double *u_prev,
                     const double *dxinv, double *partials, int nblocks, hipStream_t s) {
  hipLaunchKernelGGL(k_cfl_norm, dim3(nblocks), dim3(TB), 0, s, G, model, gamma, dt, u, u_prev, dxinv, partials);
}

bool launch_tridiag(const double *a, double *b, const double *c, double *x, int n, int ns, int *flag,
                    hipStream_t s) {
  int T, m;
  if (!team_shape(n + 1, kMaxRows, T, m)) {  // longer than one team: one thread per system
    hipLaunchKernelGGL(k_tridiag_seq, dim3(nblk(ns)), dim3(TB), 0, s, a, b, c, x, n, ns, flag);
    return true;
  }
  const long teams_per_block = TB / T;
  const long nblocks = (ns + teams_per_block - 1) / teams_per_block;
  hipLaunchKernelGGL(k_tridiag, dim3((unsigned)nblocks), dim3(TB), 0, s, a, b, c, x, n, ns, T, m, flag);
  return true;
}

void launch_dev_flux(const AosGrid &A, int model, double gamma, int dir, const double *u, double *f, hipStream_t s) {
  const long n = (long)(A.nx + 2 * A.g) * (A.ndims == 2 ? A.ny + 2 * A.g : 1);
  hipLaunchKernelGGL(k_dev_flux, dim3(nblk(n)), dim3(TB), 0, s, A, model, gamma, dir, u, f);
}

void launch_dev_upwind(const AosGrid &A, int model, int mode, double gamma, int dir, const double *uL, const double *uR,
                       const double *fL, const double *fR, const double *u, double *fI, hipStream_t s) {
  const long n = (long)((dir ? A.ny : A.nx) + 1) * (A.ndims == 2 ? (dir ? A.nx : A.ny) : 1);
  hipLaunchKernelGGL(k_dev_upwind, dim3(nblk(n)), dim3(TB), 0, s, A, model, mode, gamma, dir, uL, uR, fL, fR, u, fI);
}

void launch_dev_fd(const AosGrid &A, int dir, int par4, int bias, const double *f, double *df, hipStream_t s) {
  const int N = dir ? A.ny : A.nx, nl = A.ndims == 2 ? (dir ? A.nx : A.ny) : 1;
  const long n = (long)(N + 2 * A.g) * nl * A.nv;
  hipLaunchKernelGGL(k_dev_fd, dim3(nblk(n)), dim3(TB), 0, s, A, dir, par4, bias, f, df);
}

void launch_dev_weights(const AosGrid &A, int model, double gamma, int dir, int kind, int crweno,
                        int characteristic, int no_limiting, double eps, const double *fC, const double *u,
                        double *w1, double *w2, double *w3, long size, hipStream_t s) {
  const int N = dir ? A.ny : A.nx, nl = A.ndims == 2 ? (dir ? A.nx : A.ny) : 1;
  hipLaunchKernelGGL(k_dev_weights, dim3(nblk((long)(N + 1) * nl)), dim3(TB), 0, s, A, model, gamma, dir, kind,
                     crweno, characteristic, no_limiting, eps, fC, u, w1, w2, w3, size);
}

void launch_dev_planar(const Grid &G, const double *a, double *nat, double *tr, int to_planar, int ghosts_only,
                       double *out, hipStream_t s) {
  const long n = (long)G.nxg * G.nyg * G.nv;
  hipLaunchKernelGGL(k_dev_planar, dim3(nblk(n)), dim3(TB), 0, s, G, a, nat, tr, to_planar, ghosts_only, out);
}

hipError_t launch_pack(const Grid &G, const double *host, long q0, long np, double *u, hipStream_t s) {
  const long n = np * G.nv;
  hipLaunchKernelGGL(k_pack, dim3(nblk(n)), dim3(TB), 0, s, G, host, q0, (unsigned)n, u);
  return hipGetLastError();
}

hipError_t launch_unpack(const Grid &G, const double *u, long q0, long np, double *host, hipStream_t s) {
  const long n = np * G.nv;
  hipLaunchKernelGGL(k_unpack, dim3(nblk(n)), dim3(TB), 0, s, G, u, q0, (unsigned)n, host);
  return hipGetLastError();
}

void launch_set_time(double *time, double t, hipStream_t s) {
  hipLaunchKernelGGL(k_set_time, dim3(1), dim3(1), 0, s, time, t);
}

void launch_dev_iface(int ndims, int dir, int nx, int N, int nl, int nv, const double *src, double *dst,
                      hipStream_t s) {
  const long n = (long)(N + 1) * nl * nv;
  hipLaunchKernelGGL(k_dev_iface, dim3(nblk(n)), dim3(TB), 0, s, ndims, dir, nx, N, nl, nv, src, dst);
}

void launch_recon_only(const CaseDev *d, const Plan &pl, const CaseDev &c, int dir, int r, hipStream_t st) {
  const SweepGeom &S = dir ? c.Sy : c.Sx;
  const int what = recon_only(dir, r);
  run(K_ENDS, d, pl, what, st, nullptr, nullptr);
  for (int v = 0; v < kNRecon; v++) {
    const int cls = K_RECON + v, threads = recon_threads(kRecon[v].wide);
    if (!recon_in(S, kRecon[v].rows, kRecon[v].wide)) continue;
    // half the sweep's pairs, in blocks that all belong to the plan's only case
    const long per = threads / S.team, n = (recon_pairs(S, c.G.nv) / 2 + per - 1) / per;
    hipLaunchKernelGGL(class_kernel(pl, cls), dim3((unsigned)n), dim3(threads), 0, st, d, pl.blockcase[cls],
                       pl.firstblock[cls], what);
  }
}

void launch_class(const CaseDev *d, const Plan &pl, int cls, int s, hipStream_t st) {
  run(cls, d, pl, s, st, nullptr, nullptr);
}

void launch_weno_weights(int kind, const double *copt, const double *st, int count, double eps, double *w,
                         hipStream_t s) {
  hipLaunchKernelGGL(k_weno_weights, dim3(nblk(count)), dim3(TB), 0, s, kind, copt[0], copt[1], copt[2], st, count,
                     eps, w);
}

}  // namespace piafs
