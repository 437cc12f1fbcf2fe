// Whole steps of 1D cases in one launch.  A short line is a chain of launches
// with a few hundred values each when every pass over it is a kernel; here a
// block keeps what it works on in LDS from the first stage to the last.  The
// arithmetic is that of the kernels of a step, value by value.
#include "boundary.hpp"
#include "recon.hpp"
#include "weno.hpp"

namespace piafs {

namespace {

// the next stage's value from the solution u and the stages so far (TimeRK.c:
// 46-57), or after the last stage the new solution (:86-99); ud(j): Udot_j
template <class F>
__device__ __forceinline__ double advance(const CaseDev &C, int s, double u, F ud) {
  const int ns = C.nstages;
  if (s == ns - 1) {
    for (int j = 0; j < ns; j++) u += (C.dt * C.b[j]) * ud(j);
    return u;
  }
  for (int j = 0; j <= s; j++) {
    const double a = C.dt * C.A[(s + 1) * ns + j];
    if (a != 0.0) u += a * ud(j);
  }
  return u;
}

// CRWENO5 by components: the line couples all of its points, so one block takes
// a case, `stage` steps of it.  Bound by latency: four barriers a stage, of
// which the line solves (a wave or part of one per system, MR rows a lane) are
// the longest.  A step (RK4, Roe) in 21 launches of a graph and in this kernel, us:
//   points     8    33   128   257   258   400   513
//   launches  89    92   101   104   108   117   119
//   here      21    22    30    42    52    54    56
// The last is the longest line whose lanes' rows (8) fit a wave a system.
constexpr int kLineThreads = 768;

template <int MR, int KIND, bool LEFT>
__device__ __forceinline__ void line_system(const CaseDev &C, const double *src, int lane, int T, int *status,
                                            double *out) {
  const int N = C.Sx.N, lo = 1 + lane * MR, nlane = (N - 1) / MR;
  double A[MR], B[MR], Cc[MR], X[MR], w[MR + 5], a, b, c, x0, xN;
#pragma unroll
  for (int j = 0; j < MR + 5; j++) w[j] = lo - 3 + j <= N + 2 ? src[lo - 3 + j] : 0.0;
  assemble_rows<MR, KIND, LEFT>(C.R, w, A, B, Cc, X);
  // the end values, one on each half of the team (of two lanes or more)
  const double *e = lane < T / 2 ? src : src + N;
  row_coeffs<KIND>(0, N, LEFT, C.R, e[-3], e[-2], e[-1], e[0], e[1], e[2], a, b, c, x0);
  xN = __shfl(x0, T - 1, T);
  x0 = __shfl(x0, 0, T);
  if (lo + MR > N) {
#pragma unroll
    for (int i = 0; i < MR; i++) {
      if (lo + i >= N) {
        A[i] = 0.0;
        B[i] = 1.0;
        Cc[i] = 0.0;
        X[i] = (lo + i == N) ? xN : 0.0;
      }
    }
  }
  line_solve<MR, false>(A, B, Cc, X, lane, T, x0, nlane < T ? 0.0 : xN, nullptr, status, C.R.plain_start != 0);
  if (lane == 0) {
    out[0] = x0;
    out[N] = xN;
  }
#pragma unroll
  for (int i = 0; i < MR; i++)
    if (lo + i < N) out[lo + i] = X[i];
}

template <int MR>
__global__ void __launch_bounds__(kLineThreads) k_line(CASE_ARGS) {
  extern __shared__ double lds[];
  const CaseDev &C = cases[blockcase ? blockcase[blockIdx.x] : 0];
  constexpr int nv = kLineVars;
  const int N = C.Sx.N, ns = C.nstages, g = C.G.g, P = N + 6, tid = threadIdx.x;
  const double gam = C.P.gamma;
  double *u = lds, *U = u + nv * N + 3, *F = U + nv * P, *Ud = F + nv * P - 3, *io = Ud + ns * nv * N;
  // U, F: position i of variable v at v*P + i, i = -3 .. N+2; the interface
  // flux takes F's place when the systems are solved
  auto at = [&](int r, int v) { return io + (r * nv + v) * (N + 1); };
  for (int q = tid; q < nv * N; q += kLineThreads) {
    const int v = q / N, i = q % N;
    U[v * P + i] = u[q] = C.u[(long)v * C.G.plane + g + i];
  }
  __syncthreads();
  int T = 1;
  while (T * MR < N - 1) T <<= 1;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), per = 64 / T, groups = (2 * nv + per - 1) / per;
  const int lane = tid & (T - 1), sub = (tid & 63) / T;
  static_assert(2 * 256 + 1 + 6 <= kLineThreads, "a thread has one position at most");
  int gsrc = 0;
  double gfac = 0.0;
  const bool ghost = tid < P && (tid < 3 || tid >= N + 3), copies = ghost && ghost_copy_1d(C, tid - 3, gsrc, gfac);
  for (int step = 0; step < stage; step++)
    for (int s = 0; s < ns; s++) {
      // ghost values and the cell flux, a thread per position
      if (tid < P) {
        const int i = tid - 3;
        if (copies)
          for (int v = 0; v < nv; v++) U[v * P + i] = gfac * U[v * P + gsrc];
        else if (ghost)
          for (int v = 0; v < nv; v++)
            U[v * P + i] = ghost_value(C, v, i, 0, [&](int m, int a, int) { return U[m * P + a]; });
        point_flux(1, 0, gam, nv, [&](int m) { return U[m * P + i]; }, [&](int m, double x) { F[m * P + i] = x; });
      }
      __syncthreads();
      // uL, uR, fL, fR: a wave's teams solve systems of one bias
      for (int k = wave; k < 2 * groups; k += kLineThreads / 64) {
        const int side = k / groups, sys = (k % groups) * per + sub;
        const int sy = sys < 2 * nv ? sys : 0;  // a team past the last system repeats the first and keeps it
        const int q = sy / nv, v = sy % nv;
        const double *src = (q ? F : U) + v * P;
        double *out = at(2 * q + side, v);
#define SOLVE(KIND)                                                          \
  (side ? line_system<MR, KIND, false>(C, src, lane, T, C.status, out) \
        : line_system<MR, KIND, true>(C, src, lane, T, C.status, out))
        switch (C.R.kind) {
          case 1: SOLVE(1); break;
          case 2: SOLVE(2); break;
          case 3: SOLVE(3); break;
          default: SOLVE(0); break;
        }
#undef SOLVE
      }
      __syncthreads();
      for (int k = tid; k <= N; k += kLineThreads) {
        double uLc[3], uRc[3], a[4][3], fo[3], e[3];
#pragma unroll
        for (int m = 0; m < 3; m++) {
          uLc[m] = U[m * P + k - 1];
          uRc[m] = U[m * P + k];
#pragma unroll
          for (int r = 0; r < 4; r++) a[r][m] = at(r, m)[k];
        }
        const int mode = C.upwind;
        if (mode == 0 || mode == 3) {
          double ud[3], fs[3];
#pragma unroll
          for (int m = 0; m < 3; m++) {
            ud[m] = 0.5 * (a[1][m] - a[0][m]);
            fs[m] = 0.5 * (a[2][m] + a[3][m]);
          }
          if (mode == 0) {
            roe_e1d(gam, uLc, uRc, ud, fs, fo);
          } else {
            const double c = rusanov_e1d(gam, uLc, uRc);
            for (int m = 0; m < 3; m++) fo[m] = fs[m] - c * ud[m];
          }
        } else {
          rf_e1d(gam, mode == 2, uLc, uRc, a[0], a[1], a[2], a[3], fo, e);
        }
        for (int m = 0; m < 3; m++) F[m * P + k] = fo[m];
      }
      __syncthreads();
      for (int q = tid; q < nv * N; q += kLineThreads) {
        const int v = q / N, i = q % N;
        const double hyp = C.dxinv[g + i] * (F[v * P + i + 1] - F[v * P + i]);
        Ud[s * nv * N + q] = -hyp;
        const double x = advance(C, s, u[q], [&](int j) { return Ud[j * nv * N + q]; });
        if (s == ns - 1) u[q] = x;
        U[v * P + i] = x;
      }
      __syncthreads();
    }
  for (int q = tid; q < nv * N; q += kLineThreads) C.u[(long)(q / N) * C.G.plane + g + q % N] = u[q];
  if (tid == 0) {
    double t = *C.time;
    for (int step = 0; step < stage; step++) t = t + C.dt;
    *C.time = t;
  }
}

// The schemes without line systems: a stage reaches three points to each side,
// so a block takes a window of 63 points through all stages of a step and keeps
// the points in the middle that nothing from outside has reached.  The solution
// goes from u to Udot[0] and back (stage: 1 on the way back).  Bound by the
// latency of k_weno's chains; the windows of a line of 1024 (RK3, 51 points
// kept of 63) run side by side.  It took 46 us a step in 10 launches.
constexpr int kWin = 63;
__global__ void __launch_bounds__(256) k_tube(CASE_ARGS) {
  CASE_PREAMBLE
  (void)t;
  __shared__ Rows rows;
  constexpr int nv = kLineVars;
  __shared__ double u0[nv][kWin], U[nv][kWin + 6], Ud[4][nv][kWin], f[nv][64];
  const int N = C.Sx.N, ns = C.nstages, g = C.G.g, tid = threadIdx.x;
  const int lost = 3 * (ns - 1), core = tube_core(ns), bid = (int)(int)blockIdx.x - first;
  const int c0 = bid * core - lost;  // the window's first point
  const bool wraps = C.nzones > 0 && C.zones[0].kind == Z_PERIODIC;
  const double *src = stage ? C.Udot[0] : C.u;
  double *dst = stage ? C.u : C.Udot[0];
  auto inside = [&](int i) {  // the point a window position stands for
    if (!wraps) return min(max(i, 0), N - 1);  // beyond the ends: any value, it reaches no point kept
    const int r = i % N;
    return r < 0 ? r + N : r;
  };
  for (int q = tid; q < nv * (kWin + 6); q += 256) {
    const int v = q / (kWin + 6), p = q % (kWin + 6);
    const double x = src[(long)v * C.G.plane + g + inside(c0 + p - 3)];
    U[v][p] = x;
    if (p >= 3 && p < kWin + 3) u0[v][p - 3] = x;
  }
  // this thread's ghost value, if it has one in the window
  const int gv = tid / 6, gi = tid % 6 < 3 ? tid % 6 - 3 : N + tid % 6 - 3, gp = gi - c0 + 3;
  const bool ghost = !wraps && tid < 6 * nv && gp >= 0 && gp < kWin + 6;
  int gsrc = 0;
  double gfac = 0.0;
  const bool copies = ghost && ghost_copy_1d(C, gi, gsrc, gfac);
  for (int s = 0; s < ns; s++) {
    __syncthreads();
    if (copies) {
      U[gv][gp] = gfac * U[gv][gsrc - c0 + 3];
    } else if (ghost) {
      const int v = gv, i = gi, p = gp;
      U[v][p] = ghost_value(C, v, i, 0, [&](int m, int a, int) { return U[m][a - c0 + 3]; });
    }
    __syncthreads();
    const int x = tid & 63;
#define TUBE(KIND)                                                                                    \
  (C.R.characteristic                                                                                 \
       ? weno_tile<1, 0, KIND, true>(C, &U[0][x + 3], kWin + 6, &f[0][x], 64, true, bid & 3, rows) \
       : weno_tile<1, 0, KIND, false>(C, &U[0][x + 3], kWin + 6, &f[0][x], 64, true, bid & 3, rows))
    switch (C.R.kind) {
      case 1: TUBE(1); break;
      case 2: TUBE(2); break;
      case 3: TUBE(3); break;
      case 4: TUBE(4); break;
      default: TUBE(0); break;
    }
#undef TUBE
    __syncthreads();
    for (int q = tid; q < nv * kWin; q += 256) {
      const int v = q / kWin, k = q % kWin, i = c0 + k;
      const double hyp = C.dxinv[g + inside(i)] * (f[v][k + 1] - f[v][k]);
      Ud[s][v][k] = -hyp;
      const double x = advance(C, s, u0[v][k], [&](int j) { return Ud[j][v][k]; });
      if (s < ns - 1) {
        if (wraps || (i >= 0 && i < N)) U[v][k + 3] = x;
      } else if (k >= lost && k < lost + core && i < N) {
        dst[(long)v * C.G.plane + g + i] = x;
      }
    }
  }
  if (bid == 0 && tid == 0) *C.time = *C.time + C.dt;
}

// the solution back from Udot[0] after an odd number of steps
__global__ void __launch_bounds__(256) k_tube_back(CASE_ARGS) {
  CASE_PREAMBLE
  if (t >= (long)C.G.nx * C.G.nv) return;
  const long p = t / C.G.nx * C.G.plane + C.G.g + t % C.G.nx;
  C.u[p] = C.Udot[0][p];
}

size_t line_lds(const CaseDev &c) {
  return sizeof(double) * kLineVars * ((size_t)(1 + c.nstages) * c.G.nx + 2 * (c.G.nx + 6) + 4 * (c.G.nx + 1));
}

}  // namespace

int line_class(const CaseDev &c) {
  if (c.G.ndims != 1 || c.model != 1 || c.G.nv != kLineVars || c.cons || c.sponge || c.P.chem || c.terms != 7 || c.G.nx < 8)
    return -1;
  if (c.R.crweno) {
    if (c.R.characteristic || line_lds(c) > kLineLdsMax) return -1;
    return c.G.nx <= 4 * 64 + 1 ? K_LINE4 : c.G.nx <= 8 * 64 + 1 ? K_LINE8 : -1;
  }
  // both ends periodic, or neither
  int periodic = 0;
  for (int z = 0; z < c.nzones; z++) periodic += c.zones[z].kind == Z_PERIODIC;
  if (periodic && (periodic != 2 || c.nzones != 2 || c.zones[0].face == c.zones[1].face)) return -1;
  return K_TUBE;
}

hipError_t launch_lines(const CaseDev *d, const Plan &pl, const std::vector<CaseDev> &cases, int n, hipStream_t st,
                        MarkFn mark, void *ctx) {
  if (n <= 0) return hipSuccess;  // as the stage kernels' loops take it
  for (int cls = K_LINE4; cls <= K_LINE8; cls++) {
    if (!pl.nblocks[cls]) continue;
    size_t bytes = 0;
    for (const CaseDev &c : cases)
      if (line_class(c) == cls) bytes = line_lds(c) > bytes ? line_lds(c) : bytes;
    const KernFn k = cls == K_LINE4 ? k_line<4> : k_line<8>;
    const hipError_t e = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, kLineLdsMax);
    if (e != hipSuccess) return e;
    for (int left = n; left > 0; left -= 256) {  // a launch of bounded length
      if (mark) mark(ctx, cls, true, st);
      hipLaunchKernelGGL(k, dim3(pl.nblocks[cls]), dim3(kLineThreads), bytes, st, d, pl.blockcase[cls],
                         pl.firstblock[cls], left < 256 ? left : 256);
      if (mark) mark(ctx, cls, false, st);
    }
  }
  if (pl.nblocks[K_TUBE]) {
    auto run = [&](int cls, KernFn k, int arg) {
      if (mark) mark(ctx, cls, true, st);
      hipLaunchKernelGGL(k, dim3(pl.nblocks[cls]), dim3(256), 0, st, d, pl.blockcase[cls], pl.firstblock[cls], arg);
      if (mark) mark(ctx, cls, false, st);
    };
    for (int i = 0; i < n; i++) run(K_TUBE, k_tube, i & 1);
    if (n & 1) run(K_TUBEBACK, k_tube_back, 0);
  }
  return hipGetLastError();
}

}  // namespace piafs
