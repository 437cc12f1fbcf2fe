// Component-wise CRWENO5 reconstruction: line systems assembled and solved by
// teams of lanes.  Compiled once per segment length (RECON_ROWS rows per lane)
// and team width (RECON_WIDE: teams of 128 or 256 lanes).
#include "recon.hpp"

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
  // a species' flux is formed here from its values and the velocity, which takes one
  // plane for all of them
  const int nf = C.model == 1 ? 3 : 4;
  const bool product = C.vn_flux && q == 1 && v >= nf;
  const double *vel = (dir ? C.flux_y : C.flux_x) + (long)nf * S.plane + S.base + (long)l * S.line_stride;
  const double *src = (q == 0 || product ? (dir ? C.UT : C.U) : (dir ? C.flux_y : C.flux_x)) + (long)v * S.plane + S.base +
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
      double x = 0.0;
      if (active && pos <= hi_pos) {
        x = src[pos];
        if (product) x = vel[pos] * x;
      }
      L[slot(idx)] = x;
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
    assemble_rows<MR, KIND, LEFT>(C.R, w, A, B, Cc, X);
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
    line_solve<MR, WIDE>(A, B, Cc, X, lane, T, x0, nlane < T ? 0.0 : xN, red, C.status, C.R.plain_start != 0);
  };
  if (sides & 1) {
    solve(std::integral_constant<bool, true>(), 0);
    if (sides & 2)
#pragma unroll
      for (int i = 0; i < MR; i++) stash[i * BT + threadIdx.x] = X[i];  // this lane's own rows
  }
  if (sides & 2) solve(std::integral_constant<bool, false>(), 1);
  const Global<double> *io = dir ? C.iy : C.ix;
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
  const bool fsp = C.fuse_sp && v >= 4;
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
    // A pair of 128-lane teams has a block to itself, whose barrier has made both
    // visible.
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
        if (k > 0 && k < N) fo[k] = Lf[slot(k)] - dvv[it] * Lu[slot(k)];
      }
      if (lane < 2) {  // apart: one load for either would be a FLAT one of LDS or memory
        const int k = lane ? N : 0;
        fo[k] = io[1][line + k] - C.dsp[dir][(long)l * (N + 1) + k] * io[0][line + k];
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
  int bid = (int)blockIdx.x - first;
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
