// Ghost-point values of the boundary conditions.  Include from .hip files only.
#pragma once

#include "device.hpp"

namespace piafs {

namespace {

// ---------------------------------------------------------------------------
// Boundary conditions as a gather: each ghost point finds the last zone (in
// list order) that sets its variable and evaluates that zone's rule on the
// stage values of the interior points it reads.  The zones read interior
// points only, so list order matters only where zones overlap.
//  periodic BCPeriodic.c:22-62, extrapolate BCExtrapolate.c:16-51,
//  dirichlet BCDirichlet.c:16-45, reflect BCReflect.c:17-50, walls
//  BCSlipWall.c:24-135 / BCNoslipWall.c:22-80, BCSubsonicInflow.c:22-90,
//  BCSubsonicOutflow.c:21-78, BCSubsonicAmbivalent.c:30-125,
//  BCSupersonicInflow.c:26-80, BCSupersonicOutflow.c:25-80.
// A ghost point no zone sets keeps the value the reference never changes
// from its zero initialisation.
// ---------------------------------------------------------------------------
// does zone z set variable v (the flow BCs exist for ndims 2 only, the slip
// wall also for ndims 1; walls and outflows leave passive scalars alone)
__device__ __forceinline__ bool zone_sets(const Zone &z, int v, int ndims) {
  switch (z.kind) {
    case Z_PERIODIC: case Z_EXTRAPOLATE: case Z_DIRICHLET: case Z_REFLECT: return true;
    case Z_SPONGE: return false;
    case Z_SLIP_WALL: return ndims == 1 ? v < 3 : v < 4;
    case Z_SUBSONIC_INFLOW: case Z_SUPERSONIC_INFLOW: return ndims == 2;
    default: return ndims == 2 && v < 4;
  }
}

// value of variable v at ghost point (i, j); val(m, i, j): the stage value of
// variable m at an interior point
template <class V>
__device__ __forceinline__ double ghost_value(const CaseDev &C, int v, int i, int j, V val) {
  const Grid &G = C.G;
  const int nd = G.ndims;
  int d, face, gd, o;
  if (i < 0 || i >= G.nx) {
    d = 0; face = (i < 0) ? 1 : -1; gd = i; o = j;
    if (nd == 2 && (j < 0 || j >= G.ny)) return 0.0;  // corner: no zone reaches it
  } else {
    d = 1; face = (j < 0) ? 1 : -1; gd = j; o = i;
  }
  const int N = d ? G.ny : G.nx, od = 1 - d;
  int z = C.nzones - 1;
  for (; z >= 0; z--) {
    const Zone &Z = C.zones[z];
    if (Z.kind == Z_SPONGE || Z.dim != d || Z.face != face || !zone_sets(Z, v, nd)) continue;
    if (nd == 2 && (o < Z.is[od] || o >= Z.ie[od])) continue;
    break;
  }
  if (z < 0) return 0.0;
  const Zone &Z = C.zones[z];
  auto at = [&](int m, int a, int b) { return val(m, d ? b : a, d ? a : b); };  // (along d, across d)
  auto flow = [&](int a, int b, double u[4]) {
#pragma unroll
    for (int m = 0; m < 4; m++) u[m] = at(m, a, b);
  };
  if (Z.kind == Z_DIRICHLET) return C.bcvals[Z.vals + v];
  if (Z.kind == Z_PERIODIC) {
    // the source index across d is taken without the zone offset (BCPeriodic.c:44-52)
    const int src = (face == 1) ? gd + N : gd - N;
    return at(v, src, nd == 2 ? o - Z.is[od] : 0);
  }
  const int mir = (face == 1) ? -gd - 1 : 2 * N - gd - 1;
  const int om = nd == 2 ? o : 0;
  if (Z.kind == Z_EXTRAPOLATE) return at(v, mir, om);
  if (Z.kind == Z_REFLECT) return (-1.0) * at(v, mir, om);
  const double gam = Z.gamma, igm1 = 1.0 / (gam - 1.0);
  if (nd == 1) {  // slip wall, euler1d
    const double rho = at(0, mir, om), uvel = at(1, mir, om) / rho;
    const double energy = at(2, mir, om);
    const double pressure = (energy - 0.5 * rho * uvel * uvel) * (gam - 1.0);
    const double rg = rho, pg = pressure, ug = 2.0 * Z.vel[0] - uvel;
    if (v == 0) return rg;
    if (v == 1) return rg * ug;
    return igm1 * pg + 0.5 * rg * ug * ug;
  }
  if (v >= 4) return C.bcvals[Z.vals + v - 4];  // inflow passive scalars
  double um[4], rho, uvel, vvel, energy, pressure, rg, ug, vg, pg;
  if (Z.kind == Z_SUBSONIC_AMBIVALENT) {
    const double nx = (d == 0 ? 1.0 : 0.0) * (double)face, ny = (d == 1 ? 1.0 : 0.0) * (double)face;
    const int i1 = (face == 1) ? 0 : N - 1, i2 = (face == 1) ? 1 : N - 2;
    double u1, v1, u2, v2;
    flow(i1, o, um);
    ns2d_flowvar(um, gam, rho, u1, v1, energy, pressure);
    flow(i2, o, um);
    ns2d_flowvar(um, gam, rho, u2, v2, energy, pressure);
    const double vn = (1.5 * u1 - 0.5 * u2) * nx + (1.5 * v1 - 0.5 * v2) * ny;
    flow(mir, om, um);
    ns2d_flowvar(um, gam, rho, uvel, vvel, energy, pressure);
    if (vn > 0) { rg = Z.rho; pg = pressure; ug = Z.vel[0]; vg = Z.vel[1]; }
    else { rg = rho; pg = Z.p; ug = uvel; vg = vvel; }
  } else {
    flow(mir, om, um);
    ns2d_flowvar(um, gam, rho, uvel, vvel, energy, pressure);
    rg = rho; pg = pressure; ug = uvel; vg = vvel;  // supersonic outflow
    switch (Z.kind) {
      case Z_SLIP_WALL:
        if (d == 0) ug = 2.0 * Z.vel[0] - uvel;
        else vg = 2.0 * Z.vel[1] - vvel;
        break;
      case Z_NOSLIP_WALL:
        ug = 2.0 * Z.vel[0] - uvel;
        vg = 2.0 * Z.vel[1] - vvel;
        break;
      case Z_SUBSONIC_INFLOW: rg = Z.rho; ug = Z.vel[0]; vg = Z.vel[1]; break;
      case Z_SUBSONIC_OUTFLOW: pg = Z.p; break;
      case Z_SUPERSONIC_INFLOW: rg = Z.rho; pg = Z.p; ug = Z.vel[0]; vg = Z.vel[1]; break;
      default: break;
    }
  }
  if (v == 0) return rg;
  if (v == 1) return rg * ug;
  if (v == 2) return rg * vg;
  return igm1 * pg + 0.5 * rg * (ug * ug + vg * vg);
}

// Position i outside a line: whether its ghost values are copies of one interior
// point's in every variable; then that point, and 1 or -1 to multiply with.
// (The zone is found once; ghost_value looks for it, through dependent loads, at
// every call.)
__device__ __forceinline__ bool ghost_copy_1d(const CaseDev &C, int i, int &src, double &fac) {
  const int N = C.G.nx, face = i < 0 ? 1 : -1;
  int z = C.nzones - 1;
  for (; z >= 0; z--) {
    const Zone &Z = C.zones[z];
    if (Z.kind != Z_SPONGE && Z.dim == 0 && Z.face == face && zone_sets(Z, 0, 1)) break;
  }
  if (z < 0) return false;
  const int kind = C.zones[z].kind;
  src = kind == Z_PERIODIC ? i + face * N : face == 1 ? -i - 1 : 2 * N - i - 1;
  fac = kind == Z_REFLECT ? -1.0 : 1.0;
  return kind == Z_PERIODIC || kind == Z_EXTRAPOLATE || kind == Z_REFLECT;
}

}  // namespace

}  // namespace piafs
