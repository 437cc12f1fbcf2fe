// Device kernels of the PIAFS RHS / RK path and their host launchers.
//
// Every kernel covers a whole ensemble of cases in one launch.  Each case's
// work items are padded to whole blocks so that a block belongs to exactly
// one case: block b runs case blockcase[b], local item
// (b - firstblock[case]) * blockDim + threadIdx.  A single simulation is an
// ensemble of one.
//
// Layouts (all FP64, one plane per variable):
//   natural   : u[v*plane + (j+gy)*nxg + (i+g)]     x fastest (2D) / u[v*plane + i+g] (1D)
//   transposed: uT[v*plane + (i+g)*nyg + (j+gy)]    y fastest (2D only)
//   interface : a[(v*nlines + l)*(N+1) + k]         k = interface along the sweep (fast),
//                                                    l = interior line index
// Every sweep reads lines that are contiguous in memory: the x-sweep the
// natural state, the y-sweep the transposed copy written by the stage kernel.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

namespace piafs {

struct Grid {
  int ndims, nv, g;
  int nx, ny;        // interior sizes (ny = 1 in 1D)
  int gy;            // ghosts along y (0 in 1D)
  int nxg, nyg;      // ghosted sizes (nyg = 1 in 1D)
  long plane;        // elements per variable plane (>= nxg*nyg)
};

struct SweepGeom {
  int N;             // interior points along the sweep
  int nlines;        // interior lines
  int g;
  long plane;
  long base;         // element offset of (line 0, position 0); positions run -g .. N+g-1
  int line_stride;   // elements between consecutive lines
  int team;          // lanes sharing one line system (power of two, <= 256)
  int rows;          // interior rows (1 .. N-1) held by each lane, <= kMaxRows
  int longl;         // lines longer than one team covers (team_shape fails): their
                     // component-wise systems go through k_lrows / k_lsolve instead
};

// Longest segment of a line system one lane keeps in registers.
#ifndef PIAFS_MAX_ROWS
#define PIAFS_MAX_ROWS 16
#endif
constexpr int kMaxRows = PIAFS_MAX_ROWS;
// Doubles in the allocation-free entry point's device scratch array (32 MiB):
// piafs_tridiag_host_noalloc takes n*ns <= (capacity - 1) / 4.
#ifndef PIAFS_NOALLOC_SCRATCH_DOUBLES
#define PIAFS_NOALLOC_SCRATCH_DOUBLES ((size_t)1 << 22)
#endif
// Lane exchanges of the line-solve scans and relays by DPP (1) or by LDS
// permutes (0).
#ifndef PIAFS_SCAN_DPP
#define PIAFS_SCAN_DPP 1
#endif
// the tile kernels (k_assemble, k_stage with 32-point tiles) give each XCD a
// contiguous band of tiles (1) or take tiles in workgroup order (0)
#ifndef PIAFS_XCD_ORDER
#define PIAFS_XCD_ORDER 1
#endif
// Team shape for lines of N points: the fewest lanes (a power of two) whose
// segments of at most max_rows rows cover interior rows 1..N-1.  Returns
// false when a line is too long for one block.
bool team_shape(int N, int max_rows, int &team, int &rows);
// Lanes of the reconstruction's teams for lines of N points with `rows` rows
// per lane; false when no kernel has that shape.
bool line_shape(int N, int rows, int &team);
// Rows and team of each sweep (none longl) of one step's line systems, for its
// case's number of variables.
void choose_rows(const std::vector<SweepGeom *> &sweeps, const std::vector<int> &nvars);

// Boundary zones of boundary.inp, applied in list order: a later zone
// overwrites an earlier one where both set a variable at a ghost point.
enum ZoneKind {
  Z_PERIODIC = 0, Z_EXTRAPOLATE, Z_DIRICHLET, Z_REFLECT, Z_SPONGE, Z_NOSLIP_WALL, Z_SLIP_WALL,
  Z_SUBSONIC_INFLOW, Z_SUBSONIC_OUTFLOW, Z_SUBSONIC_AMBIVALENT, Z_SUPERSONIC_INFLOW, Z_SUPERSONIC_OUTFLOW
};
constexpr int kMaxZones = 16;
struct Zone {
  int kind, dim, face;  // face +1: the low end of dim, -1: the high end (boundary.inp)
  int is[2], ie[2];     // index box [is, ie) per dimension: the ghost layer along dim and the
                        // covered interior range across it; a sponge: a box of interior points
  int vals;             // offset of the zone's values in CaseDev::bcvals (dirichlet / sponge:
                        // nvars values; inflow: the passive scalars), -1 if none
  double rho, vel[2], p, gamma;
  double xmin, xmax;    // sponge: the zone's extent along dim
};

struct PhysParams {
  double gamma;
  // viscous (navierstokes2d)
  double inv_Re, inv_Pr, inv_gm1, Tref, T0, TS, TA, TB, two_third;
  double kappa_num;   // T0 + TA*exp(-TB/T0), constant numerator factor
  int viscous, par4;
  // derivative ghosts exchanged along dimension d (0: x, 1: y): the MPI
  // exchange of QDerivX / QDerivY that a run with more than one rank along a
  // periodic dimension performs (a no-op in a serial run)
  int xchg[2];
  // chemistry
  int chem, nflow, nlayers, z_stride;
  double k0a, k0b, k1a, k1b, k2a, k2b, k3a, k3b, k4, k5, k6;
  double q0a, q0b, q1a, q1b, q2a, q2b, q3a, q3b, q4, q5, q6;
  double ch_gm1, hnu_den, damp_coef;   // (gamma_chem - 1), c*h*nu*n_O2, dz*sO3*n_O2
  double I0, t_start_norm, t_pulse_norm;
};

struct ReconParams {
  int crweno, kind, no_limiting, characteristic;
  int plain_start;  // start the line-solve relay from trivial estimates (testing)
  double eps;
};

// A pointer to device memory in a table that kernels read.  A pointer read from
// memory is generic to the compiler: every access through it is a FLAT one, with
// its address in vector registers, and waits for LDS traffic too.  Read through
// this it is known to be global (k_next at 1024 x 1024 206 -> 193 us, 600 x 343
// 40.2 -> 35.7, 128 x 97 9.2 -> 7.9).
template <class T>
struct Global {
#ifdef __HIP_DEVICE_COMPILE__
  __attribute__((address_space(1))) T *p;
#else
  T *p;
#endif
  __host__ __device__ __forceinline__ operator T *() const { return (T *)p; }
  __host__ __device__ Global &operator=(T *q) {
    p = (decltype(p))q;
    return *this;
  }
};

// Everything a kernel needs to know about one case (device-resident table).
struct CaseDev {
  Grid G;
  SweepGeom Sx, Sy;
  int nzones, sponge;  // sponge: the case has a sponge zone
  Zone zones[kMaxZones];
  PhysParams P;
  ReconParams R;
  int model, upwind, nstages;  // upwind: 0 Roe, 1 rf-char, 2 llf-char, 3 rusanov
  int paired;    // reconstruction writes 0.5*(uR-uL), 0.5*(fL+fR) only (Roe with component-wise interpolation)
  int fuse_sp;   // species interface fluxes written by the reconstruction (set by the plan; see species_in_recon)
  int vn_flux;   // the fluxes' first species plane holds the velocity along the sweep, the reconstruction forms the
                 // species' fluxes from it (set by the plan; see velocity_for_flux)
  Global<double> dsp[2];  // per sweep and interface: Roe-average |v_n| with the entropy fix (k_flux, when fuse_sp)
  int stage_tile; // side of k_stage's transpose tiles, 32 or 64 (set by the plan)
  int unit;      // descriptor of the device-buffer operators: the interface flux in separate passes
  int terms;     // terms k_assemble adds: bit 0 hyperbolic, bit 1 parabolic, bit 2 source (7 in a step)
  double dt, A[16], b[4], c[4];
  Global<double> u, U, UT, Udot[4];
  // 2D cases of two and more stages (fused): k_next writes the next stage's
  // state itself, to Un.  The chemistry reads the stage state of other variables
  // while it does, so stage s of a case with chemistry has a buffer Us[s] apart
  // from the next one's; the other cases have one.  The descriptor table has an
  // entry of every case per stage, with U and Un those of the stage.
  int fused;
  int push[4];  // per face 2 d + (high end): ghost points that k_next copies, 1 periodic, 2 mirrored; all 0: k_ghost_next's
  Global<double> Us[4], Un;
  Global<double> flux_x, flux_y, ix[4], iy[4], fIx, fIy;
  Global<double> FV, dxinv, imap;
  Global<double> xc;      // grid coordinates with ghosts, one dimension after the other
  Global<double> bcvals;  // the zones' values (Zone::vals)
  Global<double> ends;  // paired mode: raw end-interface values of both systems of every pair [dir][pair][side][0|N]
  Global<double> time;  // current simulation time of the case; second double: the time at the start of a fused case's step
  // conservation check (conservation_check yes): boundary flux sums of each
  // stage [stage][(2 d + face) nv + v], the total boundary integral [nv], and
  // dS[d], the face element of dimension d (BoundaryIntegral.c:37-44)
  int cons;
  double dS[2];
  Global<double> bflux, tbi;
  // characteristic CRWENO5: block rows of each sweep [field][line][k] and the
  // back-substitution data of its four systems [field][system][line][k]
  Global<double> cwr[2], cwb[2];
  // sweeps of long lines: rows A, B, C and right-hand side of every system
  // [field][interface k][system], system = (line*nvars + var)*4 + r
  // (r: uL, uR, fL, fR), written by k_lrows and solved in place by k_lsolve
  Global<double> lrow[2];
  Global<int> status;   // bit 0: a zero pivot met in a line solve (tridiagLU.c:139-142 returns -1)
};

// Kernel classes launched per RK stage.  K_STAGE fills the ghost points too
// (fused cases need it at the start of a call only) and K_FLUX the line systems' end values and the viscous
// fluxes; K_GHOST, K_ENDS and K_FLUXALL (the cell fluxes of every case, those
// of K_WENO among them, which forms its own) do one thing for the operators.
// K_LINE* and K_TUBE advance 1D cases by whole steps (line.hip).
enum KClass {
  K_STAGE = 0, K_GHOST, K_FLUX, K_ENDS, K_RECON, K_LROWS = K_RECON + 10, K_LSOLVE, K_CWROWS, K_CWSOLVE, K_WENO, K_UPWIND,
  K_BFLUX, K_ASSEMBLE, K_NEXT, K_GHOSTNEXT, K_UPDATE, K_FLUXALL,
  K_LINE4, K_LINE8, K_TUBE, K_TUBEBACK,
  K_NCLASS
};
const char *kclass_name(int k);

// Block -> case tables of every kernel class for one ensemble.
struct Plan {
  int ncases = 0, nfused = 0;
  bool stage64 = false;  // k_stage with 64 x 64 tiles (every case at least 2048 x 2048)
  int nblocks[K_NCLASS] = {0};
  int *blockcase[K_NCLASS] = {nullptr};   // device arrays, one int per block (null: one case has all blocks)
  int *firstblock[K_NCLASS] = {nullptr};  // device arrays, one int per case
};

typedef void (*KernFn)(const CaseDev *, const int *, const int *, int);

// The line systems of the component-wise CRWENO5 reconstruction (recon.hip):
// one kernel, and one class K_RECON + index, per segment length and team
// width.  Narrow teams (at most 64 lanes) lie inside a wave.
struct ReconVariant {
  int rows;
  bool wide;
};
constexpr ReconVariant kRecon[] = {{4, false},  {6, false},  {8, false}, {10, false}, {12, false},
                                   {14, false}, {16, false}, {10, true}, {12, true},  {16, true}};
constexpr int kNRecon = sizeof kRecon / sizeof kRecon[0];
static_assert(K_LROWS == K_RECON + kNRecon, "a kernel class per variant");
template <int ROWS, bool WIDE>
KernFn recon_kernel();
// threads of a block: narrow teams need no more than the two that share their
// results, and small blocks leave the CU as they finish
__host__ __device__ constexpr int recon_threads(bool wide) { return wide ? 256 : 128; }
// LDS doubles of a team's line, positions -2 .. T*rows+2 with a slot unused after every `rows`
__host__ __device__ constexpr int recon_region(int T, int rows) { return T * rows + 5 + (T * rows + 5) / rows + 1; }
// of a block's: most for T = 1
__host__ __device__ constexpr int recon_line_doubles(int rows, int threads) { return threads * recon_region(1, rows); }
__host__ __device__ inline bool recon_in(const SweepGeom &S, int rows, bool wide) {
  return !S.longl && S.rows == rows && (S.team > 64) == wide;
}
__host__ __device__ inline long recon_pairs(const SweepGeom &S, int nv) { return S.longl ? 0 : (long)S.nlines * nv * 2; }
__host__ __device__ inline int recon_sweep_blocks(const SweepGeom &S, int nv) {
  const long per = recon_threads(S.team > 64) / S.team;
  return (int)((recon_pairs(S, nv) + per - 1) / per);
}
// `stage` argument that restricts a launch to reconstruction r (0 uL, 1 uR, 2
// fL, 3 fR) of one sweep
__host__ __device__ constexpr int recon_only(int dir, int r) { return (1 | (r & 1) << 1 | (r >> 1) << 2 | dir << 3) << 8; }
KernFn weno_kernel();        // k_weno (weno.hip)
constexpr int kWenoTile = 64;  // interfaces of a block

// per-class timing: called before and after each launch with the stream it goes to
typedef void (*MarkFn)(void *ctx, int cls, bool begin, hipStream_t st);

// 1D cases advanced by whole steps: the class that can take a case (-1: none;
// such a case takes the kernels of a stage), and n steps of a plan whose members
// all have one.
constexpr int kLineVars = 3;  // species come with the chemistry, which these steps leave to the others
constexpr size_t kLineLdsMax = 150 * 1024;
// points of its window a k_tube block keeps
__host__ __device__ constexpr int tube_core(int nstages) { return 63 - 6 * (nstages - 1); }
int line_class(const CaseDev &c);
hipError_t launch_lines(const CaseDev *d_cases, const Plan &plan, const std::vector<CaseDev> &cases, int n,
                        hipStream_t st, MarkFn mark, void *mark_ctx);

// Host side: blocks each case needs for each kernel class (0 = class unused).
void case_blocks(const CaseDev &c, int blocks[K_NCLASS]);
// Whether the reconstruction can write the species' Roe interface fluxes
// itself (NS2D, paired Roe, teams of 32 to 128 lanes, |v_n| buffers present).
// Lanes follow the segment length: a square case alone has such teams from 98 to
// 129 and from 162 to 2049 points a side.  A step with k_upwind writing all fluxes / with the
// reconstruction writing the species': 100 x 100 178 / 168 us, 128 x 97 185 / 173,
// 192^2 250 / 243, 256^2 338 / 332, 320^2 484 / 479, 512^2 988 / 955, 700^2 2.12 /
// 2.01 ms, 1024^2 4.10 / 3.90, 1531^2 11.62 / 11.28, 2048 x 1531 14.91 / 14.41.
// Teams of 16 lanes lost 1.4 % (256^2 with 16 rows a lane); a team of 256 lanes has
// a block to itself, without its partner.
bool species_in_recon(const CaseDev &c);
// Whether the reconstruction can form the species' cell fluxes itself, and from how
// many cells of a plan on it does: it saves k_flux traffic (1024 x 1024 133 -> 77
// us, 20 members of 96 .. 320 points a side 56 -> 45) and costs the line teams a
// load and a product a point (128 x 97: a launch of 20.8 us 0.5 us more).
constexpr long kVnFluxCells = 1L << 15;
bool velocity_for_flux(const CaseDev &c);
// Whether the case is large enough for k_stage's 64 x 64 tiles.
bool stage_tile_64(const CaseDev &c);
// doubles per interface of the characteristic CRWENO5 scratch of one sweep:
// block rows (the flow block of L, then a, b, c coefficients and the right-hand
// side of every variable of the four systems), back-substitution data (four
// systems: flow block inverse, super-diagonal block and x'; per species the
// reciprocal pivot, c and x')
int cw_row_fields(int nflow, int nv);
int cw_back_fields(int nflow, int nv);

// Stage s of the RK step for every case in the plan: stage state + BCs,
// fluxes and viscous terms, reconstruction, upwinding, assembly of Udot[s].
// Times: stage time = *time + c[s]*dt of each case.
// With `last` < K_NCLASS only the work up to that class is done (in launch
// order, which is the order of KClass), for the per-operator entry points:
// K_GHOST ends with the stage state, K_FLUX with the cell fluxes.
void launch_stage(const CaseDev *d_cases, const Plan &plan, int s, hipStream_t st, MarkFn mark, void *mark_ctx,
                  int last = K_NCLASS);
// A step: launch_begin once before the first of a call's steps, then every stage
// of each step with launch_step_stage (d_cases: the table of all stages) and
// launch_update.  Fused cases go through k_next, the others through the stage
// state, the assembly and the update u += dt*b_s*Udot_s, time += dt.
void launch_begin(const CaseDev *d_cases, const Plan &plan, hipStream_t st, MarkFn mark, void *mark_ctx);
void launch_step_stage(const CaseDev *d_cases, const Plan &plan, int s, hipStream_t st, MarkFn mark, void *mark_ctx);
void launch_update(const CaseDev *d_cases, const Plan &plan, hipStream_t st, MarkFn mark, void *mark_ctx);
// How the ghost points of each face of a case are filled (CaseDev::push).
void choose_push(CaseDev &c);

// diagnostics (single case): per-block partial max CFL and sum of squared
// step differences of the interior state
void launch_cfl_norm(const Grid &G, int model, double gamma, double dt, const double *u, const double *u_prev,
                     const double *dxinv, double *partials, int nblocks, hipStream_t s);
int cfl_norm_blocks(const Grid &G);

// Sizes of an array in the reference's layout: every point with its ghosts,
// x fastest, the nv components of a point contiguous (ny = 1 in 1D).
struct AosGrid {
  int ndims, nv, g, nx, ny;
};
// device-buffer operators on reference-layout arrays (see kernels.hip)
void launch_dev_flux(const AosGrid &A, int model, double gamma, int dir, const double *u, double *f, hipStream_t s);
void launch_dev_upwind(const AosGrid &A, int model, int mode, double gamma, int dir, const double *uL, const double *uR,
                       const double *fL, const double *fR, const double *u, double *fI, hipStream_t s);
void launch_dev_fd(const AosGrid &A, int dir, int par4, int bias, const double *f, double *df, hipStream_t s);
void launch_dev_weights(const AosGrid &A, int model, double gamma, int dir, int kind, int crweno,
                        int characteristic, int no_limiting, double eps, const double *fC, const double *u,
                        double *w1, double *w2, double *w3, long size, hipStream_t s);
// interface values of the schemes without line systems, straight between the
// reference-layout arrays (weno.hip)
void launch_dev_weno(const AosGrid &A, int model, double gamma, const ReconParams &R, int dir, bool left,
                     const double *a, const double *u, double *fI, hipStream_t s);
// ghosted reference-layout array <-> planar natural / transposed copies
void launch_dev_planar(const Grid &G, const double *a, double *nat, double *tr, int to_planar, int ghosts_only,
                       double *out, hipStream_t s);
// Interior points q0 .. q0+np-1 (x fastest) of a state: point-major values in
// pinned host memory -> the planar ghosted layout, and back.  Both say whether the
// launch failed.
hipError_t launch_pack(const Grid &G, const double *host, long q0, long np, double *u, hipStream_t s);
hipError_t launch_unpack(const Grid &G, const double *u, long q0, long np, double *host, hipStream_t s);
void launch_set_time(double *time, double t, hipStream_t s);
// one sweep's interface array: line-major -> reference layout
void launch_dev_iface(int ndims, int dir, int nx, int N, int nl, int nv, const double *src, double *dst,
                      hipStream_t s);
// reconstruction r of the systems of one sweep (not longl), end values included,
// of a plan's only case, whose descriptor is c
void launch_recon_only(const CaseDev *d_cases, const Plan &plan, const CaseDev &c, int dir, int r, hipStream_t st);
// one kernel class of stage s over the plan's cases
void launch_class(const CaseDev *d_cases, const Plan &plan, int cls, int s, hipStream_t st);

// doubles of the long-line scratch of one sweep (SweepGeom::longl)
inline size_t lrow_doubles(const SweepGeom &S, int nv) { return (size_t)4 * (S.N + 1) * S.nlines * nv * 4; }

// per-operator kernels used by the unit-level entry points
// (systems longer than one team are solved one thread per system)
// b may be overwritten (with the pivots, for systems longer than one team)
bool launch_tridiag(const double *a, double *b, const double *c, double *x, int n, int ns, int *flag,
                    hipStream_t s);
void launch_weno_weights(int kind, const double *copt, const double *st, int count, double eps, double *w,
                         hipStream_t s);

}  // namespace piafs
