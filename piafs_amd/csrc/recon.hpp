// Assembly and solution of one CRWENO5 line system by a team of lanes, MR rows
// a lane; WIDE teams span the waves of a 256-thread block, narrow ones lie in a
// wave.  Include from .hip files only.
#pragma once

#include "teams.hpp"

namespace piafs {

namespace {

// value of the team's previous (UP) or next lane; the first (last) lane of the
// team receives a value it must not use.  WIDE teams pass the wave's edge
// through red, whose two halves alternate so that one barrier suffices.
template <bool WIDE, bool UP>
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
template <bool WIDE>
__device__ __forceinline__ bool any_lane(bool p) { return WIDE ? __syncthreads_or(p) != 0 : __any(p) != 0; }

// Solves the team's system; on exit X holds the solution.  Rows: (A, B, C, X) =
// (sub-, main, super-diagonal, right-hand side).  The row before the team's
// first row is an identity row of value xfirst, the row after its last one of
// value xlast.
//
// The result is the sequential sweep of tridiagLU.c:133-150 and :243-255 bit
// for bit (see teams.hpp; for tiny numerators see the back substitution): each
// lane runs the sweep over its rows from an estimate of the state entering them,
// and entries are replaced by what the neighbour ended with until none changes.
// The estimates here use how the systems contract.  A pivot forgets its
// predecessors by a factor of about 0.1 a row, so a lane's own rows give its last
// pivot to the last bits from any start; they are run as continuants, p_k = b_k
// p_{k-1} - a_k c_{k-1} p_{k-2} with b'_k = p_k / p_{k-1}, without divisions.  x'
// and x forget by 0.55 a row or better, so the affine maps of the 64 rows before a
// segment fix its entry.  Elsewhere (weights far from optimal) the estimates are
// worse and the relays take more passes, T at most.
template <int MR, bool WIDE>
__device__ __forceinline__ void line_solve(double (&A)[MR], double (&B)[MR], double (&C)[MR], double (&X)[MR],
                                           int lane, int T, double xfirst, double xlast, double *red, int *status,
                                           bool plain_start) {
  const bool first = lane == 0, last = lane == T - 1;
  int turn = 0;
  double F[MR];
  double cin = neighbour<WIDE, true>(C[MR - 1], red, turn);
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
      const double out = neighbour<WIDE, true>(p1 * rcp_est(p0), red, turn);
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
    const double nb = neighbour<WIDE, true>(bend, red, turn);
    const bool chg = !first && !(nb == bin);
    if (!any_lane<WIDE>(chg)) break;
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
        if (!WIDE) done = !any_lane<WIDE>(!same);
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
        const double p = neighbour<WIDE, true>(y, red, turn);
        y = first ? fb : __builtin_fma(fa, p, fb);
      }
    } else {
      y = 0.0;
    }
    xin = neighbour<WIDE, true>(y, red, turn);
    if (first) xin = xfirst;
  }
  for (int it = 0; it <= T; it++) {
    double x = xin;
#pragma unroll
    for (int i = 0; i < MR; i++) x = X[i] - F[i] * x;
    const double nx = neighbour<WIDE, true>(x, red, turn);
    const bool chg = !first && !(nx == xin);
    if (!first) xin = nx;
    if (!any_lane<WIDE>(chg)) break;
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
        const double p = neighbour<WIDE, false>(y, red, turn);
        y = last ? gb : __builtin_fma(ga, p, gb);
      }
    } else {
      y = 0.0;
    }
    yin = neighbour<WIDE, false>(y, red, turn);
    if (last) yin = xlast;
  }
  // The quotients take the reciprocals at hand (wdiv's last steps): the IEEE
  // quotient's bits within its envelope.  Past the upper end of the range it
  // gives NaN where the IEEE quotient is infinite; a NaN runs on to the segment's
  // first row, and then the team divides again with the full sequence.  Numerators
  // below 2^-969, as in the tail of a species that is zero elsewhere, are not
  // looked for: there one unit in the last place can be missing (2 to 3 % of the
  // quotients of numerators below 2^-1029), and -0 becomes +0.
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
    const double ny = neighbour<WIDE, false>(x, red, turn);
    const bool chg = !last && !(ny == yin);
    if (!last) yin = ny;
    if (!any_lane<WIDE>(chg)) break;
  }
  if (any_lane<WIDE>(!(F[0] == F[0]))) {
    yin = yin0;
    for (int it = 0; it <= T; it++) {
      double x = yin;
#pragma unroll
      for (int i = MR - 1; i >= 0; i--) {
        x = (X[i] - C[i] * x) / B[i];
        F[i] = x;
      }
      const double ny = neighbour<WIDE, false>(x, red, turn);
      const bool chg = !last && !(ny == yin);
      if (!last) yin = ny;
      if (!any_lane<WIDE>(chg)) break;
    }
  }
#pragma unroll
  for (int i = 0; i < MR; i++) X[i] = F[i];
}

// Rows lo .. lo+MR-1 of a system from the line's values w[j] at positions lo-3+j
template <int MR, int KIND, bool LEFT>
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

}  // namespace

}  // namespace piafs
