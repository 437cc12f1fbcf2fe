// Component-wise CRWENO5 reconstruction: line systems assembled and solved by
// teams of lanes.  Compiled once per segment length (RECON_ROWS rows per lane)
// and team width (RECON_WIDE: teams of 128 or 256 lanes).
#include "teams.hpp"

#include <type_traits>

namespace piafs {

namespace {

constexpr int MR = RECON_ROWS;
constexpr bool WIDE = RECON_WIDE;
constexpr int BT = recon_threads(WIDE);

// ---------------------------------------------------------------------------
// Component-wise CRWENO5 reconstruction.  Systems r of a (line, variable): r =
// 0 uL, 1 uR (of the state), 2 fL, 3 fR (of the flux); r even = left-biased.  A
// team of T lanes solves the left- and right-biased systems of a pair (pair 0:
// uL, uR; pair 1: fL, fR) in turn; lane j holds rows 1 + j*MR .. of the
// interior rows 1..N-1.  Rows past N-1 are identity rows, the first of them
// (interface N, unless it follows the team) carrying the end value.
//  * weights: WENOFifthOrderCalculateWeights{JS,M,Z,YC}
//    (WENOFifthOrderCalculateWeights.c:112-237 and the variants);
//    optimal weights :202-220.
//  * row assembly: Interp1PrimFifthOrderCRWENO.c:132-201.
// Paired mode writes the two combinations the Roe upwinding uses, 0.5*(uR - uL)
// and 0.5*(fL + fR) (NavierStokes2DUpwind.c:58-60, Euler1DUpwind.c:45-52);
// split mode the four arrays.
//
// Bound by FP64 issue at two waves per SIMD, so what counts is instructions per
// row.  The operations below are the reference's, with three identities that
// keep every bit: terms that neighbouring rows share (second differences and
// their squares, candidate sums) are formed once; 2, 4 and 1/4 scale exactly,
// so a product with one of them joins the following sum in one fma; and
// 2/3 * w = 2 * RN(1/3 * w).  The other parts of the gain are line_solve's
// cheaper estimates, quotients of the back substitution from reciprocals the
// estimates leave, and passes without per-row exits.  Blocks are two waves, so
// that LDS is given back as they finish.  1024 x 1024, nv 11: 254 -> about 175
// VALU instructions per row and system, 222 registers, 1025 -> 748 us a launch;
// 20 uneven cases of 96 .. 320 points a side (segment lengths to fit their
// lines, see choose_rows) 774 -> 361 us of reconstruction a stage.
// ---------------------------------------------------------------------------

// value of the team's previous (UP) or next lane; the first (last) lane of the
// team receives a value it must not use.  WIDE teams pass the wave's edge
// through red, whose two halves alternate so that one barrier suffices.
template <bool UP>
__device__ __forceinline__ double neighbour(double v, double *red, int &turn) {
  double r = lane_step<UP>(v);
  if (WIDE) {
    const int wave = (int)threadIdx.x >> 6, x = (int)threadIdx.x & 63;
    double *e = red + 4 * (turn++ & 1);
    if (x == (UP ? 63 : 0)) e[wave] = v;
    __syncthreads();
    if (x == (UP ? 0 : 63)) r = e[(wave + (UP ? 3 : 1)) & 3];
  }
  return r;
}

// true on every lane when p holds on any lane of the wave (WIDE: block)
__device__ __forceinline__ bool any_lane(bool p) { return WIDE ? __syncthreads_or(p) != 0 : __any(p) != 0; }

// Solves the team's system; on exit X holds the solution.  Rows: (A, B, C, X) =
// (sub-, main, super-diagonal, right-hand side).  The row before the team's
// first row is an identity row of value xfirst, the row after its last one of
// value xlast.
//
// The result is the sequential sweep of tridiagLU.c:133-150 and :243-255 bit
// for bit (see teams.hpp): each lane runs the sweep over its rows from an
// estimate of the state entering them, and entries are replaced by what the
// neighbour ended with until none changes.  The estimates here use how the
// systems contract.  A pivot forgets its predecessors by a factor of about 0.1
// a row, so a lane's own rows give its last pivot to the last bits from any
// start; they are run as continuants, p_k = b_k p_{k-1} - a_k c_{k-1} p_{k-2}
// with b'_k = p_k / p_{k-1}, without divisions.  x' and x forget by 0.55 a row
// or better, so the affine maps of the 64 rows before a segment fix its entry.
// Elsewhere (weights far from optimal) the estimates are worse and the relays
// take more passes, T at most.
__device__ __forceinline__ void line_solve(double (&A)[MR], double (&B)[MR], double (&C)[MR], double (&X)[MR],
                                           int lane, int T, double xfirst, double xlast, double *red, int *status,
                                           bool plain_start) {
  const bool first = lane == 0, last = lane == T - 1;
  int turn = 0;
  double F[MR];
  double cin = neighbour<true>(C[MR - 1], red, turn);
  if (first) cin = 0.0;
  // pivot entering the segment
  double bin = first ? 1.0 : 0.5;
  if (!plain_start) {
    constexpr int rounds = MR >= 12 ? 1 : MR >= 6 ? 2 : 3;
#pragma unroll 1
    for (int r = 0; r < rounds; r++) {
      double p0 = 1.0, p1 = bin;
#pragma unroll
      for (int i = 0; i < MR; i++) {
        const double ac = A[i] * (i == 0 ? cin : C[i > 0 ? i - 1 : 0]);
        const double p2 = __builtin_fma(B[i], p1, -(ac * p0));
        p0 = p1;
        p1 = p2;
      }
      const double out = neighbour<true>(p1 * rcp_est(p0), red, turn);
      if (!first) bin = out;
    }
  } else if (!first) {
    bin = 1.0;
  }
  // multipliers, then the relay of the pivots: a segment whose entry changed
  // derives them again until one repeats (all that follow repeat with it)
  double bend = bin;
  {
    double c = cin;
#pragma unroll
    for (int i = 0; i < MR; i++) {
      F[i] = wdiv(A[i], bend);
      bend = B[i] - F[i] * c;
      c = C[i];
    }
  }
  for (int it = 0; it <= T; it++) {
    const double nb = neighbour<true>(bend, red, turn);
    const bool chg = !first && !(nb == bin);
    if (!any_lane(chg)) break;
    if (!first) bin = nb;
    double b = bin, c = cin;
    bool done = false;
#pragma unroll
    for (int i0 = 0; i0 < MR; i0 += 2) {
      if (!done) {  // uniform
        bool same = true;
#pragma unroll
        for (int i = i0; i < i0 + 2; i++) {
          const double f = wdiv(A[i], b);
          same = __double_as_longlong(f) == __double_as_longlong(F[i]);
          F[i] = f;
          b = B[i] - f * c;
          c = C[i];
        }
        if (!WIDE) done = !any_lane(!same);
      }
    }
    if (!done) bend = b;
  }
  // x' entering the segment: affine map of the segment, then the maps of the
  // segments before it
  double xin;
  {
    double fa = 1.0, fb = first ? xfirst : 0.0;
#pragma unroll
    for (int i = 0; i < MR; i++) {
      fa = fa * F[i];
      fb = __builtin_fma(-F[i], fb, X[i]);
    }
    if (MR & 1) fa = -fa;
    double y = fb;
    if (!plain_start) {
      constexpr int back = (64 + MR - 1) / MR;
      const int n = back < T - 1 ? back : T - 1;
#pragma unroll 1
      for (int j = 0; j < n; j++) {
        const double p = neighbour<true>(y, red, turn);
        y = first ? fb : __builtin_fma(fa, p, fb);
      }
    } else {
      y = 0.0;
    }
    xin = neighbour<true>(y, red, turn);
    if (first) xin = xfirst;
  }
  for (int it = 0; it <= T; it++) {
    double x = xin;
#pragma unroll
    for (int i = 0; i < MR; i++) x = X[i] - F[i] * x;
    const double nx = neighbour<true>(x, red, turn);
    const bool chg = !first && !(nx == xin);
    if (!first) xin = nx;
    if (!any_lane(chg)) break;
  }
  // b' and x' of every row, in the reference's arithmetic
  double small = fabs(bin);
  {
    double b = bin, x = xin, c = cin;
#pragma unroll
    for (int i = 0; i < MR; i++) {
      b = B[i] - F[i] * c;
      x = X[i] - F[i] * x;
      c = C[i];
      small = fmin(small, fabs(b));
      B[i] = b;
      X[i] = x;
    }
  }
  if (small == 0.0) atomicOr(status, 1);
  // back substitution: entries from above likewise
  double (&rb)[MR] = A;
  double yin;
  {
    double ga = 1.0, gb = last ? xlast : 0.0;
#pragma unroll
    for (int i = MR - 1; i >= 0; i--) {
      rb[i] = rcp_est(B[i]);
      ga = ga * (C[i] * rb[i]);
      gb = __builtin_fma(-C[i], gb, X[i]) * rb[i];
    }
    if (MR & 1) ga = -ga;
    double y = gb;
    if (!plain_start) {
      constexpr int back = (64 + MR - 1) / MR;
      const int n = back < T - 1 ? back : T - 1;
#pragma unroll 1
      for (int j = 0; j < n; j++) {
        const double p = neighbour<false>(y, red, turn);
        y = last ? gb : __builtin_fma(ga, p, gb);
      }
    } else {
      y = 0.0;
    }
    yin = neighbour<false>(y, red, turn);
    if (last) yin = xlast;
  }
  // The quotients take the reciprocals at hand (wdiv's last steps): the IEEE
  // quotient's bits within its envelope.  Past the ends of the range it gives
  // NaN where the IEEE quotient is infinite; a NaN runs on to the segment's
  // first row, and then the team divides again with the full sequence.
  const double yin0 = yin;
  for (int it = 0; it <= T; it++) {
    double x = yin;
#pragma unroll
    for (int i = MR - 1; i >= 0; i--) {
      const double n = X[i] - C[i] * x;
      const double q = n * rb[i];
      x = __builtin_fma(__builtin_fma(-B[i], q, n), rb[i], q);
      F[i] = x;
    }
    const double ny = neighbour<false>(x, red, turn);
    const bool chg = !last && !(ny == yin);
    if (!last) yin = ny;
    if (!any_lane(chg)) break;
  }
  if (any_lane(!(F[0] == F[0]))) {
    yin = yin0;
    for (int it = 0; it <= T; it++) {
      double x = yin;
#pragma unroll
      for (int i = MR - 1; i >= 0; i--) {
        x = (X[i] - C[i] * x) / B[i];
        F[i] = x;
      }
      const double ny = neighbour<false>(x, red, turn);
      const bool chg = !last && !(ny == yin);
      if (!last) yin = ny;
      if (!any_lane(chg)) break;
    }
  }
#pragma unroll
  for (int i = 0; i < MR; i++) X[i] = F[i];
}

// Rows lo .. lo+MR-1 of a system from the line's values w[j] at positions lo-3+j
template <int KIND, bool LEFT>
__device__ __forceinline__ void assemble_rows(const ReconParams &R, const double *__restrict__ w, double (&A)[MR],
                                              double (&B)[MR], double (&C)[MR], double (&X)[MR]) {
  const double s6 = 1.0 / 6.0, s56 = 5 * s6, t3 = 1.0 / 3.0, t1312 = 13.0 / 12.0, q14 = 1.0 / 4.0;
  const double c1 = 0.2, c2 = 0.5, c3 = 0.3;
  // second difference around w[j+1], in the bias's order, scaled and squared
  auto curv = [&](int j) {
    const double d = LEFT ? __builtin_fma(-2.0, w[j + 1], w[j]) + w[j + 2] : __builtin_fma(-2.0, w[j + 1], w[j + 2]) + w[j];
    return t1312 * d * d;
  };
  // s6 and 5 s6 times the values at w[i+2] (A), w[i+3] (B) and, right-biased, w[i+4]
  double ta = curv(LEFT ? 0 : 1), tb = curv(LEFT ? 1 : 2);
  double pA = s6 * w[2], qA = s56 * w[2], pB = s6 * w[3], qB = s56 * w[3];
  double shared = LEFT ? s6 * w[1] + qA : qA + pB;  // a candidate that is the next row's too
#pragma unroll
  for (int i = 0; i < MR; i++) {
    const double m3 = LEFT ? w[i] : w[i + 5], m2 = LEFT ? w[i + 1] : w[i + 4], m1 = LEFT ? w[i + 2] : w[i + 3];
    const double p1 = LEFT ? w[i + 3] : w[i + 2], p2 = LEFT ? w[i + 4] : w[i + 1];
    const double tc = curv(LEFT ? i + 2 : i + 3);
    const double pC = s6 * w[i + 4], qC = s56 * w[i + 4];
    const double next = LEFT ? pA + qB : qB + pC;
    const double f1 = LEFT ? shared : next, f2 = LEFT ? qA + pB : pA + qB, f3 = LEFT ? next : shared;
    shared = next;
    pA = pB;
    qA = qB;
    pB = pC;
    qB = qC;
    double a1 = c1, a2 = c2, a3 = c3;
    if (!R.no_limiting) {
      const double r3 = 3 * m1;
      const double e1 = __builtin_fma(-4.0, m2, m3) + r3, e2 = m2 - p1, e3 = __builtin_fma(-4.0, p1, r3) + p2;
      const double b1 = __builtin_fma(q14, e1 * e1, LEFT ? ta : tc), b2 = __builtin_fma(q14, e2 * e2, tb),
                   b3 = __builtin_fma(q14, e3 * e3, LEFT ? tc : ta);
      const double t = KIND == 3 ? m3 - 4 * m2 + 6 * m1 - 4 * p1 + p2 : 0.0;
      weno_of<KIND>(c1, c2, c3, b1, b2, b3, t, R.eps, a1, a2, a3);
    }
    ta = tb;
    tb = tc;
    const double t1 = t3 * a1, t2 = t3 * a2, t3a = t3 * a3;
    const double lo = __builtin_fma(2.0, t1, t2);
    B[i] = __builtin_fma(2.0, t3a, __builtin_fma(2.0, t2, t1));
    A[i] = LEFT ? lo : t3a;
    C[i] = LEFT ? t3a : lo;
    X[i] = a1 * f1 + a2 * f2 + a3 * f3;
    __builtin_amdgcn_sched_barrier(0);  // a row at a time: interleaved rows need twice the registers
  }
}

// A team's region of the staged lines: line position p (-2 .. T*MR+2) at slot
// p + 2, one unused slot after every MR (even), so that lanes reading their
// windows, MR apart, hit different banks.
static_assert(MR % 2 == 0, "segments have an even number of rows");
__device__ __forceinline__ int slot(int i) { return i + i / MR; }

// sides: bit 0 the left-biased system, bit 1 the right-biased one
template <int KIND>
__device__ __forceinline__ void recon_pair(const CaseDev &C, int dir, long sys, bool active, int sides, int lane,
                                           double *red, double *stash, double *lines, unsigned *arrived) {
  const SweepGeom &S = dir ? C.Sy : C.Sx;
  const int nv = C.G.nv, N = S.N, nl = S.nlines, g = S.g, T = S.team;
  const long sy = active ? sys : 0;
  const int q = (int)(sy % 2), v = (int)((sy / 2) % nv), l = (int)((sy / 2) / nv);
  const double *src = (q == 0 ? (dir ? C.UT : C.U) : (dir ? C.flux_y : C.flux_x)) + (long)v * S.plane + S.base +
                      (long)l * S.line_stride;
  const long line = ((long)v * nl + l) * (N + 1);
  const int lo = 1 + lane * MR;
  const int hi_pos = N + g - 1;
  const double *ends = C.ends + 4 * ((dir ? recon_pairs(C.Sx, nv) : 0) + sy);
  double *L = lines + (threadIdx.x / T) * recon_region(T, MR);
  // species pairs whose two teams are different waves (T = 64) meet through
  // an arrival counter per pair, cleared before any wave can reach it
  if (!WIDE && C.fuse_sp && T == 64) {
    if (threadIdx.x < BT / 128) arrived[threadIdx.x] = 0u;
    __syncthreads();
  }
  auto sync = [&]() {  // all lanes of the team have finished their LDS accesses before any lane goes on
    if (WIDE) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
  };
  // the line, positions -2 .. T*MR+2 (zero past its last ghost), read by
  // consecutive lanes: both systems of the pair take their windows from it
  const int tot = T * MR + 5;
  for (int b = 0; b < tot; b += T) {
    const int idx = b + lane;
    if (idx < tot) {
      const int pos = idx - 2;
      L[slot(idx)] = (active && pos <= hi_pos) ? src[pos] : 0.0;
    }
  }
  sync();
  const int nlane = (N - 1) / MR;  // the lane holding row N
  double X[MR];
  auto solve = [&](auto left_c, int side) {
    constexpr bool LEFT = decltype(left_c)::value;
    double x0 = 0.0, xN = 0.0;
    if (active && lane == 0) x0 = ends[2 * side];
    if (active && lane == (nlane < T ? nlane : T - 1)) xN = ends[2 * side + 1];
    double A[MR], B[MR], Cc[MR], w[MR + 5];
#pragma unroll
    for (int j = 0; j < MR + 5; j++) w[j] = L[lane * (MR + 1) + j + j / MR];  // positions lo-3 .. lo+MR+1
    assemble_rows<KIND, LEFT>(C.R, w, A, B, Cc, X);
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
    line_solve(A, B, Cc, X, lane, T, x0, nlane < T ? 0.0 : xN, red, C.status, C.R.plain_start != 0);
  };
  if (sides & 1) {
    solve(std::integral_constant<bool, true>(), 0);
    if (sides & 2)
#pragma unroll
      for (int i = 0; i < MR; i++) stash[i * BT + threadIdx.x] = X[i];  // this lane's own rows
  }
  if (sides & 2) solve(std::integral_constant<bool, false>(), 1);
  double *const *io = dir ? C.iy : C.ix;
  if (!C.paired) {  // interior interfaces of uL, uR / fL, fR apart
    for (int side = sides == 2 ? 1 : 0; side < (sides == 1 ? 1 : 2); side++) {
      sync();  // the windows, or the side before, are read
#pragma unroll
      for (int i = 0; i < MR; i++)
        L[lane * (MR + 1) + (i + 1) + (i + 1) / MR] = (sides == 3 && side == 0) ? stash[i * BT + threadIdx.x] : X[i];
      sync();
      double *out = io[2 * q + side] + line;
      for (int b = 1; b < N; b += T) {
        const int k = b + lane;
        if (active && k < N) out[k] = L[slot(k)];
      }
    }
    return;
  }
  // a species of a case whose reconstruction writes the species fluxes: the
  // |v_n| of this lane's interfaces, loaded now so that the combination step
  // below hides their latency (the line's N + 1 <= T MR + 2 interfaces take at
  // most MR + 2 per lane)
  constexpr int KO = MR + 2;
  const bool fsp = !WIDE && C.fuse_sp && v >= 4;
  double dvv[KO];
#pragma unroll
  for (int it = 0; it < KO; it++) dvv[it] = 0.0;
  if (fsp && (T == 64 || q == 1)) {  // a team of at most 32 lanes writes when it is the flux team
    const double *dv = C.dsp[dir] + (long)l * (N + 1);
#pragma unroll
    for (int it = 0; it < KO; it++) {
      const int k = it * T + lane;
      if (active && k <= N) dvv[it] = dv[k];
    }
  }
  sync();  // every window of the team is read
#pragma unroll
  for (int i = 0; i < MR; i++) {
    const double xl = stash[i * BT + threadIdx.x];
    L[lane * (MR + 1) + (i + 1) + (i + 1) / MR] = q ? 0.5 * (xl + X[i]) : 0.5 * (X[i] - xl);
  }
  sync();
  if (fsp) {
    // A species: its Roe flux f_I = 0.5 (fL + fR) - |v_n| 0.5 (uR - uL), the
    // upwinder's arithmetic, is written here from the combinations of the
    // pair's two teams (u and f sources of one line and species), which sit
    // side by side in the block.  A team of at most 32 lanes shares its wave
    // with its partner, so the wave's own LDS sync has made both visible and
    // the flux team writes.  Teams of 64 lanes are two waves: each publishes
    // its combination with a release increment of the pair's counter, and the
    // one that arrives second (acquire) writes, so neither waits.  The two end
    // interfaces take the combinations k_recon_ends wrote.
    bool writer = q == 1;
    if (T == 64) {
      unsigned prev = 0u;
      if (lane == 0)
        prev = __hip_atomic_fetch_add(&arrived[(threadIdx.x >> 6) >> 1], 1u, __ATOMIC_ACQ_REL,
                                      __HIP_MEMORY_SCOPE_WORKGROUP);
      writer = __shfl(prev, 0, 64) == 1u;
    }
    if (writer && active) {
      const double *Lp = lines + ((threadIdx.x / T) ^ 1) * recon_region(T, MR);
      const double *Lf = q ? L : Lp, *Lu = q ? Lp : L;
      double *fo = (dir ? C.fIy : C.fIx) + line;
#pragma unroll
      for (int it = 0; it < KO; it++) {
        const int k = it * T + lane;
        if (k <= N) {
          const bool end = k == 0 || k == N;
          const double fs = end ? io[1][line + k] : Lf[slot(k)];
          const double ud = end ? io[0][line + k] : Lu[slot(k)];
          fo[k] = fs - dvv[it] * ud;
        }
      }
    }
    return;
  }
  double *out = io[q] + line;
  for (int b = 1; b < N; b += T) {
    const int k = b + lane;
    if (active && k < N) out[k] = L[slot(k)];
  }
}

// Blocks hold BT / T whole teams; a block never mixes sweeps.  A case's sweeps
// whose lines have this segment length and team width, or, when `stage` carries
// a recon_only() selection, one system of every pair of one sweep and source.
__global__ void __attribute__((amdgpu_flat_work_group_size(BT, BT), amdgpu_waves_per_eu(2)))
k_recon(CASE_ARGS) {
  CASE_PREAMBLE
  const int only = stage >> 8;
  if ((stage & 0xFF) >= C.nstages) return;
  __shared__ double red[8];
  __shared__ double stash[MR * BT];
  __shared__ double lines[recon_line_doubles(MR, BT)];
  __shared__ unsigned arrived[2];
  int bid = (int)(blockIdx.x - firstblock[cidx]);
  int dir = 0, sides = 3;
  if (only) {
    dir = (only >> 3) & 1;
    sides = 1 << ((only >> 1) & 1);
  } else {
    const int nbx = recon_in(C.Sx, MR, WIDE) ? recon_sweep_blocks(C.Sx, C.G.nv) : 0;
    if (bid >= nbx) {
      dir = 1;
      bid -= nbx;
    }
  }
  const SweepGeom &S = dir ? C.Sy : C.Sx;
  const int T = S.team;
  const int lane = threadIdx.x & (T - 1);
  long sys = (long)bid * (BT / T) + threadIdx.x / T;
  if (only) sys = 2 * sys + ((only >> 2) & 1);
  const bool active = sys < recon_pairs(S, C.G.nv);
  switch (C.R.kind) {
    case 1: recon_pair<1>(C, dir, sys, active, sides, lane, red, stash, lines, arrived); break;
    case 2: recon_pair<2>(C, dir, sys, active, sides, lane, red, stash, lines, arrived); break;
    case 3: recon_pair<3>(C, dir, sys, active, sides, lane, red, stash, lines, arrived); break;
    default: recon_pair<0>(C, dir, sys, active, sides, lane, red, stash, lines, arrived); break;
  }
}

}  // namespace

template <>
KernFn recon_kernel<RECON_ROWS, RECON_WIDE>() { return k_recon; }

}  // namespace piafs
