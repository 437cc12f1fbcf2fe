// Tridiagonal systems solved by teams of lanes.  Include from .hip files only.
#pragma once

#include "device.hpp"

namespace piafs {

namespace {

// ---------------------------------------------------------------------------
// Tridiagonal line systems solved by teams of lanes, with the reference's
// arithmetic.
//
// A team of T lanes (a power of two; teams of more than 64 lanes span whole
// waves of one block) owns one system, and each lane keeps a segment of at
// most kMaxRows consecutive rows in registers.  The result is the one of the
// sequential Thomas sweep of tridiagLU.c:133-150 (fac = a_k/b'_{k-1},
// b'_k = b_k - fac c_{k-1}, x'_k = x_k - fac x'_{k-1}) and :243-255
// (x_k = (x'_k - c_k x_{k+1}) / b'_k), bit for bit:
//  1. each segment gets an estimate of the state entering it -- the pivot
//     b' from a scan of the segments' Moebius maps b'_{k-1} -> b'_k (2x2
//     matrices), x' from a scan of their affine maps;
//  2. every lane runs the sweep over its rows from its entry state, and each
//     lane's entry becomes the state its predecessor ended with; this repeats
//     until no entry changes.  Lane 0 starts from the exact state, so the
//     fixed point is reached after at most T passes and is exactly the
//     sequential sweep; with the estimates (and the sweep's contraction) the
//     ends are usually exact after the first pass, so two passes are typical;
//  3. the back substitution is treated the same way from the top.
// The systems are never written to memory; only the solution is.
// ---------------------------------------------------------------------------
struct Mob {
  double a, b, c, d;  // [[a, b], [c, d]]
};
struct Aff {
  double a, b;  // x -> a*x + b
};

// Rescale by a power of two (exact) so that products of many segment maps
// neither overflow nor underflow; a Moebius map is unchanged by scaling.
__device__ __forceinline__ Mob mob_norm(Mob r) {
  const double mx = fmax(fmax(fabs(r.a), fabs(r.b)), fmax(fabs(r.c), fabs(r.d)));
  if (mx > 0.0 && mx < INFINITY) {
    const int e = ilogb(mx);
    r.a = ldexp(r.a, -e);
    r.b = ldexp(r.b, -e);
    r.c = ldexp(r.c, -e);
    r.d = ldexp(r.d, -e);
  }
  return r;
}
__device__ __forceinline__ Mob mob_mul(const Mob &x, const Mob &y) {
  Mob r;
  r.a = x.a * y.a + x.b * y.c;
  r.b = x.a * y.b + x.b * y.d;
  r.c = x.c * y.a + x.d * y.c;
  r.d = x.c * y.b + x.d * y.d;
  return mob_norm(r);
}
// outer o inner
__device__ __forceinline__ Aff aff_cmp(const Aff &o, const Aff &i) { return Aff{o.a * i.a, o.a * i.b + o.b}; }

// Lane moves of a double by DPP (a VALU operand modifier, no LDS round trip):
// lanes without a source (or outside ROWMASK) keep their own value.  CTRL:
// row_shr:d 0x110+d and row_shl:d 0x100+d move within rows of 16 lanes,
// wave_shr:1 0x138 and wave_shl:1 0x130 across the wave, row_bcast:15 0x142
// and row_bcast:31 0x143 broadcast a row's last lane to the following rows.
template <int CTRL, int ROWMASK = 0xF>
__device__ __forceinline__ double dpp_move(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int l0 = (int)(unsigned)b, h0 = (int)(unsigned)(b >> 32);
  const int lo = __builtin_amdgcn_update_dpp(l0, l0, CTRL, ROWMASK, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(h0, h0, CTRL, ROWMASK, 0xF, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
template <int CTRL, int ROWMASK = 0xF>
__device__ __forceinline__ Mob dpp_mob(const Mob &x) {
  return Mob{dpp_move<CTRL, ROWMASK>(x.a), dpp_move<CTRL, ROWMASK>(x.b), dpp_move<CTRL, ROWMASK>(x.c),
             dpp_move<CTRL, ROWMASK>(x.d)};
}
template <int CTRL, int ROWMASK = 0xF>
__device__ __forceinline__ Aff dpp_aff(const Aff &x) {
  return Aff{dpp_move<CTRL, ROWMASK>(x.a), dpp_move<CTRL, ROWMASK>(x.b)};
}
// value of lane i-1 (UP) or i+1 of the wave
template <bool UP>
__device__ __forceinline__ double lane_step(double v) {
  return UP ? dpp_move<0x138>(v) : dpp_move<0x130>(v);
}

// Exclusive scans over the lanes of a team.  `lane` is the lane within the
// team; `red` is LDS for one Mob per wave of the block.
__device__ Mob team_scan_mob(Mob x, int lane, int T, double *red) {
  const int W = T < 64 ? T : 64;
  const int wl = lane & (W - 1);
#if PIAFS_SCAN_DPP
  // within rows of 16 lanes (a team of fewer lanes lies inside one row), then
  // across the rows of the wave from each row's last lane
  const int rl = wl & 15;
  if (W > 1) { const Mob o = dpp_mob<0x111>(x); if (rl >= 1) x = mob_mul(x, o); }
  if (W > 2) { const Mob o = dpp_mob<0x112>(x); if (rl >= 2) x = mob_mul(x, o); }
  if (W > 4) { const Mob o = dpp_mob<0x114>(x); if (rl >= 4) x = mob_mul(x, o); }
  if (W > 8) { const Mob o = dpp_mob<0x118>(x); if (rl >= 8) x = mob_mul(x, o); }
  if (W > 16) { const Mob o = dpp_mob<0x142, 0xA>(x); if (wl & 16) x = mob_mul(x, o); }
  if (W > 32) { const Mob o = dpp_mob<0x143, 0xC>(x); if (wl & 32) x = mob_mul(x, o); }
#else
  for (int d = 1; d < W; d <<= 1) {
    Mob o;
    o.a = __shfl_up(x.a, d, W);
    o.b = __shfl_up(x.b, d, W);
    o.c = __shfl_up(x.c, d, W);
    o.d = __shfl_up(x.d, d, W);
    if (wl >= d) x = mob_mul(x, o);
  }
#endif
  Mob pre = {1.0, 0.0, 0.0, 1.0};
  if (T > 64) {
    const int w = lane >> 6, wave = threadIdx.x >> 6;
    if (wl == 63) {
      double *s = red + 4 * wave;
      s[0] = x.a; s[1] = x.b; s[2] = x.c; s[3] = x.d;
    }
    __syncthreads();
    for (int k = 0; k < w; k++) {
      const double *s = red + 4 * (wave - w + k);
      pre = mob_mul(Mob{s[0], s[1], s[2], s[3]}, pre);
    }
    __syncthreads();
  }
  Mob e;
#if PIAFS_SCAN_DPP
  e = Mob{lane_step<true>(x.a), lane_step<true>(x.b), lane_step<true>(x.c), lane_step<true>(x.d)};
#else
  e.a = __shfl_up(x.a, 1, W);
  e.b = __shfl_up(x.b, 1, W);
  e.c = __shfl_up(x.c, 1, W);
  e.d = __shfl_up(x.d, 1, W);
#endif
  if (wl == 0) e = pre;
  else if (T > 64) e = mob_mul(e, pre);
  return e;
}

__device__ Aff team_scan_aff_fwd(Aff x, int lane, int T, double *red) {
  const int W = T < 64 ? T : 64;
  const int wl = lane & (W - 1);
#if PIAFS_SCAN_DPP
  const int rl = wl & 15;
  if (W > 1) { const Aff o = dpp_aff<0x111>(x); if (rl >= 1) x = aff_cmp(x, o); }
  if (W > 2) { const Aff o = dpp_aff<0x112>(x); if (rl >= 2) x = aff_cmp(x, o); }
  if (W > 4) { const Aff o = dpp_aff<0x114>(x); if (rl >= 4) x = aff_cmp(x, o); }
  if (W > 8) { const Aff o = dpp_aff<0x118>(x); if (rl >= 8) x = aff_cmp(x, o); }
  if (W > 16) { const Aff o = dpp_aff<0x142, 0xA>(x); if (wl & 16) x = aff_cmp(x, o); }
  if (W > 32) { const Aff o = dpp_aff<0x143, 0xC>(x); if (wl & 32) x = aff_cmp(x, o); }
#else
  for (int d = 1; d < W; d <<= 1) {
    const Aff o = {__shfl_up(x.a, d, W), __shfl_up(x.b, d, W)};
    if (wl >= d) x = aff_cmp(x, o);
  }
#endif
  Aff pre = {1.0, 0.0};
  if (T > 64) {
    const int w = lane >> 6, wave = threadIdx.x >> 6;
    if (wl == 63) {
      red[2 * wave] = x.a;
      red[2 * wave + 1] = x.b;
    }
    __syncthreads();
    for (int k = 0; k < w; k++) pre = aff_cmp(Aff{red[2 * (wave - w + k)], red[2 * (wave - w + k) + 1]}, pre);
    __syncthreads();
  }
#if PIAFS_SCAN_DPP
  Aff e = {lane_step<true>(x.a), lane_step<true>(x.b)};
#else
  Aff e = {__shfl_up(x.a, 1, W), __shfl_up(x.b, 1, W)};
#endif
  if (wl == 0) e = pre;
  else if (T > 64) e = aff_cmp(e, pre);
  return e;
}

__device__ Aff team_scan_aff_bwd(Aff x, int lane, int T, double *red) {
  const int W = T < 64 ? T : 64;
  const int wl = lane & (W - 1);
#if PIAFS_SCAN_DPP
  // within rows of 16 lanes, then from the first lane of the following rows
  // (no DPP broadcast runs backwards: two LDS permutes)
  const int rl = wl & 15, rw = W < 16 ? W : 16;
  if (W > 1) { const Aff o = dpp_aff<0x101>(x); if (rl + 1 < rw) x = aff_cmp(x, o); }
  if (W > 2) { const Aff o = dpp_aff<0x102>(x); if (rl + 2 < rw) x = aff_cmp(x, o); }
  if (W > 4) { const Aff o = dpp_aff<0x104>(x); if (rl + 4 < rw) x = aff_cmp(x, o); }
  if (W > 8) { const Aff o = dpp_aff<0x108>(x); if (rl + 8 < rw) x = aff_cmp(x, o); }
  if (W > 16) {
    const int src = ((int)(threadIdx.x & 63) | 15) + 1;  // first lane of the next row
    const Aff o = {__shfl(x.a, src & 63, 64), __shfl(x.b, src & 63, 64)};
    if (!(wl & 16)) x = aff_cmp(x, o);
  }
  if (W > 32) {
    const Aff o = {__shfl(x.a, 32, 64), __shfl(x.b, 32, 64)};
    if (!(wl & 32)) x = aff_cmp(x, o);
  }
#else
  for (int d = 1; d < W; d <<= 1) {
    const Aff o = {__shfl_down(x.a, d, W), __shfl_down(x.b, d, W)};
    if (wl + d < W) x = aff_cmp(x, o);
  }
#endif
  Aff suf = {1.0, 0.0};
  if (T > 64) {
    const int w = lane >> 6, nw = T >> 6, wave = threadIdx.x >> 6;
    if (wl == 0) {
      red[2 * wave] = x.a;
      red[2 * wave + 1] = x.b;
    }
    __syncthreads();
    for (int k = nw - 1; k > w; k--) suf = aff_cmp(Aff{red[2 * (wave - w + k)], red[2 * (wave - w + k) + 1]}, suf);
    __syncthreads();
  }
#if PIAFS_SCAN_DPP
  Aff e = {lane_step<false>(x.a), lane_step<false>(x.b)};
#else
  Aff e = {__shfl_down(x.a, 1, W), __shfl_down(x.b, 1, W)};
#endif
  if (wl == W - 1) e = suf;
  else if (T > 64) e = aff_cmp(e, suf);
  return e;
}

// (a, b) of the previous lane of the team (dir = +1) or of the next one
// (dir = -1); the first (last) lane of the team keeps its own values.
__device__ __forceinline__ void team_shift2(double &a, double &b, int lane, int T, int dir, double *red) {
  const int W = T < 64 ? T : 64;
  const int wl = lane & (W - 1);
  double pa, pb;
#if PIAFS_SCAN_DPP
  // across team boundaries too: a team's first (last) lane receives another
  // team's value, which it does not use
  if (dir > 0) {
    pa = lane_step<true>(a);
    pb = lane_step<true>(b);
  } else {
    pa = lane_step<false>(a);
    pb = lane_step<false>(b);
  }
#else
  if (dir > 0) {
    pa = __shfl_up(a, 1, W);
    pb = __shfl_up(b, 1, W);
  } else {
    pa = __shfl_down(a, 1, W);
    pb = __shfl_down(b, 1, W);
  }
#endif
  if (T > 64) {
    const int wave = threadIdx.x >> 6;
    const bool edge_out = dir > 0 ? (wl == 63) : (wl == 0);
    if (edge_out) {
      red[2 * wave] = a;
      red[2 * wave + 1] = b;
    }
    __syncthreads();
    const bool edge_in = dir > 0 ? (wl == 0 && lane != 0) : (wl == 63 && lane != T - 1);
    if (edge_in) {
      pa = red[2 * (wave - dir)];
      pb = red[2 * (wave - dir) + 1];
    }
    __syncthreads();
  }
  a = pa;
  b = pb;
}

// true on every lane of the wave (T <= 64) or block (T > 64) when `p` holds
// on any of them
__device__ __forceinline__ bool team_any(bool p, int T) {
  if (T > 64) return __syncthreads_or(p) != 0;
  return __any(p) != 0;
}

// v_rcp_f64 refined by two Newton steps: a reciprocal good to the last bits,
// used only for the estimates that start the exact passes
__device__ __forceinline__ double rcp_est(double b) {
  double r = __builtin_amdgcn_rcp(b);
  r = fma(r, fma(-b, r, 1.0), r);
  r = fma(r, fma(-b, r, 1.0), r);
  return r;
}

// Forward elimination of team_solve: on exit B holds b' and X holds x' of
// every row, Fk the multipliers.  The row before the team's first row has
// pivot bfirst, super-diagonal cfirst and x' xfirst (an identity row: 1, 0,
// its value).  zp is set when a pivot is zero.
template <int MR>
__device__ __forceinline__ void team_forward(double (&A)[MR], double (&B)[MR], double (&Cc)[MR], double (&X)[MR],
                                             double (&Fk)[MR], int n, int lane, int T, double bfirst, double cfirst,
                                             double xfirst, double *red, bool plain_start, bool &zp) {
  const bool has = n > 0;
  double cin = 0.0, unused = 0.0;
#pragma unroll
  for (int i = 0; i < MR; i++)
    if (i == n - 1) cin = Cc[i];
  team_shift2(cin, unused, lane, T, +1, red);
  if (lane == 0) cin = cfirst;
  // pivot entering the segment: scan of M_k = [[b_k, -a_k c_{k-1}], [1, 0]] on (b'_{k-1}, 1)
  Mob P = {1.0, 0.0, 0.0, 1.0};
#pragma unroll
  for (int i = 0; i < MR; i++) {
    if (i < n) {
      const double ac = A[i] * (i == 0 ? cin : Cc[i > 0 ? i - 1 : 0]);
      const Mob R = {B[i] * P.a - ac * P.c, B[i] * P.b - ac * P.d, P.a, P.b};
      P = R;
    }
  }
  P = mob_norm(P);
  const Mob E = team_scan_mob(P, lane, T, red);
  double bin = lane == 0 ? bfirst : (plain_start ? 1.0 : (E.a + E.b) / (E.c + E.d));
  // multipliers along the estimated pivots; affine maps of x'
  double bend = bin;
  Aff F = {lane == 0 ? 0.0 : 1.0, lane == 0 ? xfirst : 0.0};
  {
    double c = cin;
#pragma unroll
    for (int i = 0; i < MR; i++) {
      if (i < n) {
        const double fac = A[i] / bend;
        bend = B[i] - fac * c;
        c = Cc[i];
        Fk[i] = fac;
        F = Aff{-(fac * F.a), X[i] - fac * F.b};
      } else {
        Fk[i] = 0.0;
      }
    }
  }
  const Aff Ef = team_scan_aff_fwd(F, lane, T, red);
  double xin = lane == 0 ? xfirst : (plain_start ? 0.0 : Ef.a * xfirst + Ef.b);
  // relay of segment ends until every entry equals its predecessor's end
  for (int it = 0;; it++) {
    double xend = xin;
#pragma unroll
    for (int i = 0; i < MR; i++)
      if (i < n) xend = X[i] - Fk[i] * xend;
    double nb = bend;
    team_shift2(nb, xend, lane, T, +1, red);
    const bool bchg = lane != 0 && !(nb == bin);
    const bool changed = has && lane != 0 && (bchg || !(xend == xin));
    if (lane != 0) {
      bin = nb;
      xin = xend;
    }
    if (!team_any(changed, T) || it > T) break;
    if (bchg) {  // pivots of this segment derived again from the new entry, until they repeat
      const double bend_old = bend;
      double c = cin, bb = bin;
      bool live = true;
#pragma unroll
      for (int i = 0; i < MR; i++) {
        if (i < n && live) {
          const double fac = A[i] / bb;
          if (__double_as_longlong(fac) == __double_as_longlong(Fk[i])) {
            live = false;  // same multiplier, so the same pivot here and in every later row
          } else {
            bb = B[i] - fac * c;
            c = Cc[i];
            Fk[i] = fac;
          }
        }
      }
      bend = live ? bb : bend_old;
    }
  }
  // b' and x' of every row, in the reference's arithmetic
  zp = zp || ((bin == 0.0) && has);
  {
    double b = bin, x = xin, c = cin;
#pragma unroll
    for (int i = 0; i < MR; i++) {
      if (i < n) {
        b = B[i] - Fk[i] * c;
        x = X[i] - Fk[i] * x;
        c = Cc[i];
        zp = zp || (b == 0.0);
        B[i] = b;
        X[i] = x;
      }
    }
  }
}

// Back substitution of team_solve: B holds b', X holds x' of every row; on
// exit X holds the solution.  The row after the team's last row (held by the
// lane with is_last) has solution xlast.  W is scratch.
template <int MR>
__device__ __forceinline__ void team_backward(double (&B)[MR], double (&Cc)[MR], double (&X)[MR], double (&W)[MR],
                                              int n, int lane, int T, bool is_last, double xlast, double *red,
                                              bool plain_start) {
  const bool has = n > 0;
  // estimate of x entering from above, then the relay
  Aff Gm = {is_last ? 0.0 : 1.0, is_last ? xlast : 0.0};
#pragma unroll
  for (int i = MR - 1; i >= 0; i--) {
    if (i < n) {
      const double rb = rcp_est(B[i]);
      Gm = Aff{-(Cc[i] * rb) * Gm.a, (X[i] - Cc[i] * Gm.b) * rb};
    }
  }
  const Aff Eb = team_scan_aff_bwd(Gm, lane, T, red);
  double yin = is_last ? xlast : (plain_start ? 0.0 : Eb.a * xlast + Eb.b);
  for (int it = 0;; it++) {
    double xv = yin, dummy = 0.0;
    bool live = true;
#pragma unroll
    for (int i = MR - 1; i >= 0; i--) {
      if (i < n && live) {
        const double nx = (X[i] - Cc[i] * xv) / B[i];
        // from the second pass on: a row that repeats its value leaves every row above unchanged
        if (it > 0 && __double_as_longlong(nx) == __double_as_longlong(W[i])) live = false;
        W[i] = nx;
        xv = nx;
      }
    }
    if (n > 0) xv = W[0];
    team_shift2(xv, dummy, lane, T, -1, red);
    const bool changed = has && !is_last && !(xv == yin);
    if (!is_last) yin = xv;
    if (!team_any(changed, T) || it > T) break;
  }
#pragma unroll
  for (int i = 0; i < MR; i++)
    if (i < n) X[i] = W[i];
}

// Solve one team's system.  On entry the n rows of this lane hold
// (A, B, Cc, X) = (sub-, main, super-diagonal, right-hand side); on exit X
// holds the solution and B the pivots.  The row before the team's first row
// is an identity row carrying xfirst; the row after the team's last row (held
// by the lane with is_last) is one carrying xlast.  Every lane of every team
// of the block must call this (it may synchronise the block).
// The multipliers of the
// pivot chain (fac = a_k / b'_{k-1}, one division each) are kept per row, so
// the x' chain of a pass costs no division: every pass takes the segments'
// entry states, runs the x' chain along the kept multipliers, and relays the
// segment ends; only when an entry pivot changes are the multipliers derived
// again.  Once no entry changes, one pass without divisions writes b' and x'
// (fac * c and fac * x' exactly as the reference computes them).  The back
// substitution iterates the same way from the top.  If `plain_start` is set
// the scanned estimates are replaced by the trivial ones (b' = 1, x' = 0), so
// that the relay runs through many passes (testing).
template <int MR>
__device__ __forceinline__ void team_solve(double (&A)[MR], double (&B)[MR], double (&Cc)[MR], double (&X)[MR],
                                                int n, int lane, int T, bool is_last, double xfirst, double xlast,
                                                double *red, int *status, bool plain_start) {
  double Fk[MR];
  bool zp = false;
  team_forward<MR>(A, B, Cc, X, Fk, n, lane, T, 1.0, 0.0, xfirst, red, plain_start, zp);
  team_backward<MR>(B, Cc, X, Fk, n, lane, T, is_last, xlast, red, plain_start);
  if (zp) atomicOr(status, 1);
}

}  // namespace

}  // namespace piafs
