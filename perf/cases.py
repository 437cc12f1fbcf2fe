"""Performance cases: what a program that uses this framework has it do, with
the sizes of its own decks, tests and benchmark, through the public entry
points of ``piafs_amd``.

A case is a dict of plain values; ``prepare`` makes what a program holds before
the call (decks read, handles open, inputs in memory), ``run`` is one pass,
``work`` the bytes and operations one pass cannot do without, and ``exact`` the
same pass in plain 64-bit torch, without this repository's kernels.

Kinds:
  solve      a state handed to a resident case, advanced some steps, read back
             (``set_solution``, ``set_time``, ``step``, ``solution``)
  rhs        one right-hand side of a host state (``rhs``)
  operators  one hyperbolic evaluation and the state's derivatives through the
             device-buffer operators, on torch tensors and a torch stream
  ensemble   many cases of uneven sizes advanced together (``Batch``)
"""
from __future__ import annotations

import math
import os
import tempfile

import numpy as np
import torch

import piafs_amd
from piafs_amd import decks

GHOSTS = 3
DX = 10.0 * math.pi / 1024  # grid spacing of the photochemistry decks


def listed():
    return [
        # the smallest call: a short 1D line (the density wave of the tests),
        # CRWENO5 components, where launches and latency count
        dict(name="sine_128", kind="solve", deck="sine", nx=128, ny=1, steps=50),
        # the plain method at its own size: Sod tube, characteristic WENO5, SSPRK3
        dict(name="sod_1024", kind="solve", deck="sod", nx=1024, ny=1, steps=60),
        # a small photochemistry solve, as most served requests and ensemble
        # members are
        dict(name="photochem_128x97", kind="solve", deck="photochem", nx=128, ny=97, steps=20, scheme="crweno5",
             weights="js", Re=1000.0),
        # an ordinary ragged one with WENO5 components
        dict(name="photochem_600x343_weno5", kind="solve", deck="photochem", nx=600, ny=343, steps=12, scheme="weno5",
             weights="js", Re=1000.0),
        # the headline configuration, 1024 x 1024 CRWENO5
        dict(name="photochem_1024", kind="solve", deck="photochem", nx=1024, ny=1024, steps=10, scheme="crweno5",
             weights="js", Re=1000.0),
        # the largest: lines of two and more waves, an odd side
        dict(name="photochem_2048x1531", kind="solve", deck="photochem", nx=2048, ny=1531, steps=4, scheme="crweno5",
             weights="js", Re=1000.0),
        # the shipped Riemann problem: characteristic mapped WENO5, rf-char,
        # SSPRK3, inviscid, mirror boundaries
        dict(name="riemann_201", kind="solve", deck="riemann", nx=201, ny=201, steps=25),
        # the shipped jet's shape: photochemistry, characteristic WENO5,
        # rf-char, supersonic in- and outflow, viscous
        dict(name="jet_500x100", kind="solve", deck="jet", nx=500, ny=100, steps=15),
        # one right-hand side for a program that keeps its own time integrator
        dict(name="rhs_512x385", kind="rhs", deck="photochem", nx=512, ny=385, scheme="crweno5", weights="js",
             Re=1000.0),
        # the function-table drop-in: each operator on the caller's device arrays
        dict(name="operators_384x250", kind="operators", deck="photochem", nx=384, ny=250, scheme="crweno5",
             weights="js", Re=1000.0),
        # an ensemble of uneven sides, WENO5 and CRWENO5 mixed
        dict(name="ensemble_20", kind="ensemble", count=20, lo=96, hi=320, mix=7, steps=3),
        # the shipped lid-driven cavity: linear upwind interpolation, no-slip walls
        dict(name="cavity_128", kind="solve", deck="cavity", nx=128, ny=128, steps=25),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["photochem", "photochem", "photochem", "tube", "char", "rhs", "operators", "ensemble"])
    if kind == "tube":
        if rng.random() < 0.5:
            return dict(kind="solve", deck="sine", nx=_log_int(rng, 64, 1500), ny=1, steps=rng.randint(20, 60))
        return dict(kind="solve", deck="sod", nx=_log_int(rng, 128, 4000), ny=1, steps=rng.randint(20, 60))
    if kind == "char":
        which = rng.choice(["riemann", "jet", "cavity"])
        if which != "jet":
            n = _log_int(rng, 65, 500)
            return dict(kind="solve", deck=which, nx=n, ny=n, steps=rng.randint(5, 25))
        return dict(kind="solve", deck="jet", nx=_log_int(rng, 100, 600), ny=_log_int(rng, 60, 500),
                    steps=rng.randint(4, 15))
    if kind == "ensemble":
        return dict(kind="ensemble", count=rng.randint(6, 24), lo=rng.randint(64, 110), hi=rng.randint(180, 320),
                    mix=rng.randint(0, 1000), steps=rng.randint(2, 4))
    top = 1100 if kind == "photochem" else 520
    nx, ny = _log_int(rng, 64, top), _log_int(rng, 64, top)
    case = dict(kind="solve" if kind == "photochem" else kind, deck="photochem", nx=nx, ny=ny,
                scheme=rng.choice(["crweno5", "crweno5", "weno5"]), weights=rng.choice(["js", "js", "mapped", "z"]),
                Re=round(math.exp(rng.uniform(math.log(1e2), math.log(5e3))), 1))
    if kind == "photochem":
        case["steps"] = max(3, min(20, int(6e6 / (nx * ny))))
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _developed(u, nx, ny, seed):
    """A photochemistry state some way into a run: the deck's perturbed gas
    with slow smooth motion, the beam's heating, ozone spent under the beam and
    the excited species it leaves."""
    r = np.random.default_rng(seed)
    ph = r.uniform(0, 2 * math.pi, 4)
    x = 2 * math.pi * np.arange(nx) / nx
    y = (2 * math.pi * np.arange(ny) / ny)[:, None]
    vx = 0.02 * np.sin(x + ph[0]) * np.cos(y + ph[1])
    vy = 0.02 * np.cos(2 * x + ph[2]) * np.sin(y + ph[3])
    beam = np.exp(np.cos(x - math.pi) + np.cos(y - math.pi) - 2.0)
    q = u.reshape(ny, nx, -1)
    rho = q[..., 0]
    q[..., 1] = rho * vx
    q[..., 2] = rho * vy
    q[..., 3] = q[..., 3] * (1.0 + 0.01 * beam) + 0.5 * rho * (vx * vx + vy * vy)
    q[..., 5] *= 1.0 - 0.1 * beam
    for m, a in ((6, 1e-6), (7, 1e-4), (8, 1e-5), (9, 5e-5)):
        q[..., m] = a * beam * (1.0 + 0.01 * r.uniform(-1, 1, (ny, nx)))
    return u


def _deck(case, seed):
    """The deck of a case with its state of this seed."""
    nx, ny = case["nx"], case["ny"]
    kind = case["deck"]
    r = np.random.default_rng(seed)
    if kind == "sine":
        dk = decks.density_sine_1d(N=nx, n_iter=case["steps"], dt=0.25 / nx)
        k = r.integers(1, 3)
        x = np.arange(nx) / nx
        rho = 1.0 + 0.1 * np.sin(2 * math.pi * (k * x + r.random())) + 0.02 * np.sin(6 * math.pi * (x + r.random()))
        dk.u[:, 0] = rho
        dk.u[:, 1] = rho
        dk.u[:, 2] = (1.0 / 1.4) / 0.4 + 0.5 * rho
    elif kind == "sod":
        dk = decks.sod_1d(N=nx, n_iter=None)
        a = r.uniform(0.9, 1.1, 4)
        left = np.arange(nx) < (nx - 1) // 2
        dk.u[:, 0] = np.where(left, a[0], 0.125 * a[1])
        dk.u[:, 2] = np.where(left, a[2], 0.1 * a[3]) / 0.4
    elif kind == "riemann":
        dk = decks.riemann_2d(N=nx, dt=0.2 / nx)
        dk.u *= 1.0 + 0.02 * r.uniform(-1, 1)
        dk.u[:, 0] *= 1.0 + 1e-3 * r.uniform(-1, 1, nx * ny)
    elif kind == "jet":
        inflow = ("supersonic-inflow", 1, 1, -1e99, 1e99, 0, 0, 1.0, 0.0, 1.6, 0.7071, 1.0, 0.01, 0.0, 0.0, 0.0, 0.0,
                  0.0)
        bc = [("periodic", 0, 1, 0, 0, -1e99, 1e99), ("periodic", 0, -1, 0, 0, -1e99, 1e99), inflow,
              ("supersonic-outflow", 1, -1, -1e99, 1e99, 0, 0)]
        dk = decks.ns2d_open_box(nx=nx, ny=ny, dt=0.005, boundary=bc, flow=(1.0, 0.0, 1.6, None), seed=seed,
                                 scheme="weno5", interp="characteristic", upwinding="rf-char", Re=150.0,
                                 include_chemistry=True, L=(nx - 1) * DX)
    elif kind == "cavity":
        walls = [("noslip-wall", d, f, *((0, 0, -1e99, 1e99) if d == 0 else (-1e99, 1e99, 0, 0)),
                  0.1 if (d, f) == (1, -1) else 0.0, 0.0) for d in (0, 1) for f in (1, -1)]
        dk = decks.ns2d_open_box(nx=nx, ny=ny, dt=0.64 / nx, boundary=walls, flow=(1.0, 0.0, 0.0, None), bump=0.0,
                                 seed=seed, scheme="upw5", Re=3200.0, L=1.0)
        X, Y = np.meshgrid(*dk.x, indexing="xy")  # a rotating start
        vx, vy = 0.1 * (Y - 0.5).reshape(-1), -0.1 * (X - 0.5).reshape(-1)
        rho = dk.u[:, 0]
        dk.u[:, 1], dk.u[:, 2] = rho * vx, rho * vy
        dk.u[:, 3] += 0.5 * rho * (vx * vx + vy * vy)
    else:
        Re = case["Re"]
        dk = decks.ns2d_photochem(nx=nx, ny=ny, n_iter=case.get("steps", 1), dt=decks.stable_dt(Re), seed=seed,
                                  scheme=case["scheme"], weights=case["weights"], Re=Re, dx=DX, L=nx * DX)
        _developed(dk.u, nx, ny, seed)
    return dk


def _members(case, seed):
    """Ensemble members: sizes and schemes from the case, states from the seed."""
    ms = decks.ensemble(n=case["count"], seed=1000 * (case["mix"] + 1), n_iter=200, side=(case["lo"], case["hi"]),
                        Re_range=(1e2, 1e3))
    for k, m in enumerate(ms):
        nx, ny = m.deck.dims
        r = np.random.default_rng([seed, k])
        m.deck.u[:, 0] = 1.0 + 1e-3 * r.uniform(-1, 1, nx * ny)
        _developed(m.deck.u, nx, ny, seed + k)
    return [m.deck for m in ms]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        with tempfile.TemporaryDirectory() as d:
            dirs = [dk.write(os.path.join(d, str(k))) for k, dk in enumerate(_members(case, seed))]
            batch = piafs_amd.Batch(dirs)
        return dict(kind=kind, batch=batch, steps=case["steps"])
    dk = _deck(case, seed)
    with tempfile.TemporaryDirectory() as d:
        c = piafs_amd.Case(dk.write(d))
    state = dict(kind=kind, case=c, u=np.ascontiguousarray(dk.u), steps=case.get("steps", 0))
    if kind == "operators":
        state.update(_operator_buffers(case, dk))
    return state


def _operator_buffers(case, dk):
    """The caller's device arrays: the ghosted state (interior filled) and the
    outputs, in the layouts the operators take."""
    nx, ny, nv, g = case["nx"], case["ny"], dk.nvars, GHOSTS
    u = torch.zeros(ny + 2 * g, nx + 2 * g, nv, dtype=torch.float64)
    u[g:-g, g:-g] = torch.from_numpy(dk.u).reshape(ny, nx, nv)
    u = u.cuda()
    out = {"u": u}
    for d, shape in ((0, (ny, nx + 1, nv)), (1, (ny + 1, nx, nv))):
        out["f%d" % d] = torch.zeros_like(u)
        out["du%d" % d] = torch.zeros_like(u)
        for name in ("uL", "uR", "fL", "fR", "fI"):
            out["%s%d" % (name, d)] = torch.zeros(shape, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    return dict(buf=out, stream=torch.cuda.Stream())


def run(state):
    kind = state["kind"]
    if kind == "ensemble":
        b = state["batch"]
        b.step(state["steps"])
        return [b.solution(k) for k in b.slots]
    c = state["case"]
    if kind == "rhs":
        return c.rhs(state["u"], 0.45)
    if kind == "operators":
        b, st = state["buf"], state["stream"].cuda_stream
        p = {k: t.data_ptr() for k, t in b.items()}
        c.dev_boundary_fill(p["u"], 0.45, st)
        for d in (0, 1):
            c.dev_flux(p["u"], d, p["f%d" % d], st)
            for name, upw, uflag in (("uL", 1, 1), ("uR", -1, 1), ("fL", 1, 0), ("fR", -1, 0)):
                c.dev_interp_interfaces(p["%s%d" % (name, d)], p["u"] if uflag else p["f%d" % d], p["u"], upw, d,
                                        uflag, st)
            c.dev_upwind(p["fI%d" % d], p["fL%d" % d], p["fR%d" % d], p["uL%d" % d], p["uR%d" % d], p["u"], d, 0.45,
                         st)
            c.dev_first_derivative_par(p["du%d" % d], p["u"], d, 1, st)
        return b
    c.set_solution(state["u"])
    c.set_time(0.0)
    c.step(state["steps"])
    return c.solution()


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _rates(deck, scheme):
    """variables, RK stages, dimensions, and operations per variable, dimension
    and stage of a cell: four reconstructions (weights, rows, line solve) and
    the flux, upwinding and divergence."""
    nv, stages, nd = {"sine": (3, 4, 1), "sod": (3, 3, 1), "riemann": (4, 3, 2), "jet": (11, 4, 2),
                      "cavity": (4, 4, 2), "photochem": (11, 4, 2)}[deck]
    per = 4 * (95 if scheme == "crweno5" else 9 if deck == "cavity" else 70) + 40
    return nv, stages, nd, per


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        nbytes = flops = 0.0
        for dk in _members(case, 0):
            w = work(dict(kind="solve", deck="photochem", nx=dk.dims[0], ny=dk.dims[1],
                          scheme=dk.solver["hyp_space_scheme"], steps=case["steps"]))
            nbytes += w["bytes"]
            flops += w["flops"]
        return {"bytes": nbytes, "flops": flops}
    nv, stages, nd, per = _rates(case["deck"], case.get("scheme", "weno5"))
    cells = float(case["nx"] * case["ny"])
    state = 8.0 * nv * cells
    if kind == "rhs":  # the state in, its right-hand side out
        return {"bytes": 2 * state, "flops": cells * nv * nd * per}
    if kind == "operators":
        # per dimension: flux (read, write), four interpolations (read, write),
        # upwinding (five reads, one write), derivative (read, write)
        return {"bytes": state * (2 + nd * (2 + 8 + 6 + 2)), "flops": cells * nv * nd * per}
    # a step reads and writes the solution once; the state comes in and goes out
    return {"bytes": 2 * state * (case["steps"] + 1), "flops": case["steps"] * stages * cells * nv * nd * per}


# ---------------------------------------------------------------------------
# the same pass in plain 64-bit torch
# ---------------------------------------------------------------------------
def _weights(kind, c, m3, m2, m1, p1, p2, eps=1e-6):
    """WENO5 nonlinear weights (Jiang-Shu, mapped, Borges Z) for optimal weights c."""
    b = (13.0 / 12.0 * (m3 - 2 * m2 + m1) ** 2 + 0.25 * (m3 - 4 * m2 + 3 * m1) ** 2,
         13.0 / 12.0 * (m2 - 2 * m1 + p1) ** 2 + 0.25 * (m2 - p1) ** 2,
         13.0 / 12.0 * (m1 - 2 * p1 + p2) ** 2 + 0.25 * (3 * m1 - 4 * p1 + p2) ** 2)
    if kind == "z":
        tau = (b[2] - b[0]).abs()
        a = [ck * (1 + (tau / (bk + eps)) ** 2) for ck, bk in zip(c, b)]
    else:
        a = [ck / (bk + eps) ** 2 for ck, bk in zip(c, b)]
    s = a[0] + a[1] + a[2]
    w = [x / s for x in a]
    if kind == "mapped":
        a = [x * (ck + ck * ck - 3 * ck * x + x * x) / (ck * ck + x * (1 - 2 * ck)) for ck, x in zip(c, w)]
        s = a[0] + a[1] + a[2]
        w = [x / s for x in a]
    return w


def _weno5(kind, m3, m2, m1, p1, p2):
    w = _weights(kind, (0.1, 0.6, 0.3), m3, m2, m1, p1, p2)
    return (w[0] * (2 * m3 - 7 * m2 + 11 * m1) + w[1] * (-m2 + 5 * m1 + 2 * p1)
            + w[2] * (2 * m1 + 5 * p1 - p2)) / 6


def _stencil(q, left):
    """Five values of every interface of lines q[..., N + 2 g]."""
    n = q.shape[-1] - 2 * GHOSTS + 1
    s = [q[..., k:k + n] for k in range(6)]
    return s[:5] if left else s[:0:-1]


def _line_values(q, left, crweno, kind):
    """Interface values of lines q[..., N + 2 g], WENO5 or the compact scheme
    (WENO5 values at the two end interfaces)."""
    m3, m2, m1, p1, p2 = _stencil(q, left)
    if kind == "linear":
        return (2 * m3 - 13 * m2 + 47 * m1 + 27 * p1 - 3 * p2) / 60
    w5 = _weno5(kind, m3, m2, m1, p1, p2)
    if not crweno:
        return w5
    w = _weights(kind, (0.2, 0.5, 0.3), m3, m2, m1, p1, p2)
    x = (w[0] * (m2 + 5 * m1) + w[1] * (5 * m1 + p1) + w[2] * (m1 + 5 * p1)) / 6
    lo, hi = (2 * w[0] + w[1]) / 3, w[2] / 3
    b = (w[0] + 2 * w[1] + 2 * w[2]) / 3
    a, c = (lo, hi) if left else (hi, lo)
    n = q.shape[-1] - 2 * GHOSTS
    a, b, c, x = (t.movedim(-1, 0).contiguous() for t in (a, b, c, x))
    w5 = w5.movedim(-1, 0)
    x[0], x[n] = w5[0], w5[n]
    b[0] = b[n] = 1.0
    a[0] = a[n] = c[0] = c[n] = 0.0
    for k in range(1, n + 1):
        f = a[k] / b[k - 1]
        b[k] -= f * c[k - 1]
        x[k] -= f * x[k - 1]
    x[n] /= b[n]
    for k in range(n - 1, -1, -1):
        x[k] = (x[k] - c[k] * x[k + 1]) / b[k]
    return x.movedim(0, -1)


class _Plain:
    """The right-hand side and time step of a deck in torch, FP64."""

    def __init__(self, dk):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        s, ph = dk.solver, dk.physics
        self.dims = dk.dims + [1] * (2 - len(dk.dims))
        self.nx, self.ny = self.dims
        self.nd, self.nv = len(dk.dims), dk.nvars
        self.nf = 3 if self.nd == 1 else 4
        self.zone_gamma = self.gamma = ph.get("gamma", 1.4)
        self.crweno = s["hyp_space_scheme"] == "crweno5"
        self.char = s["hyp_interp_type"] == "characteristic"
        self.upw = ph["upwinding"]
        self.kind = "mapped" if dk.weno.get("mapped") else "z" if dk.weno.get("borges") else "js"
        if s["hyp_space_scheme"] == "upw5":
            self.kind = "linear"
        self.rk, self.dt, self.boundary = s["time_scheme_type"], s["dt"], dk.boundary
        self.inv = []
        for x in dk.x:
            e = np.concatenate([[2 * x[0] - x[1]], x, [2 * x[-1] - x[-2]]])
            d = 2.0 / (e[2:] - e[:-2])
            self.inv.append(torch.from_numpy(np.concatenate([[d[0]] * GHOSTS, d, [d[-1]] * GHOSTS])).to(self.dev))
        self.Re, self.Pr, self.Tref = ph.get("Re", -1.0), ph.get("Pr", 0.72), 273.15
        self.chem = dk.chemistry is not None
        if self.chem:
            self._chemistry(dk)

    def _chemistry(self, dk):
        ch = dk.chemistry
        NA, kB, e, c_light, h = 6.02214076e23, 1.380649e-23, 1.60217663e-19, 3.0e8, 6.62607015e-34
        Ptot, Ti = ch["Ptot"], 288.0
        t_pulse, F0 = 1e-8, 2000.0
        R = NA * kB / 0.032
        g = self.gamma = 918.45 / 650.0
        mu = 1.99e-5 * math.exp(1.5 * math.log(Ti / 275.0)) * (275.0 + 110.4) / (Ti + 110.4)
        kap = 2.70e-2 * math.exp(1.5 * math.log(Ti / 275.0)) * (275.0 + 245.4 * math.exp(-27.6 / 275.0)) / (
            Ti + 245.4 * math.exp(-27.6 / Ti))
        lam = 2.48e-7
        kg = 2 * (2 * math.pi / lam) * math.sin(0.17 * math.pi / 180)
        n = Ptot / (kB * Ti)
        cs = math.sqrt(g * R * Ti)
        rho = Ptot / (R * Ti)
        self.Tref = Ti
        self.Re, self.Pr = rho * cs / kg / mu, g * R / (g - 1) * mu / kap
        rate = kg * cs / n
        k = dict(k0a=0.9 * 3.3e-13, k0b=0.1 * 3.3e-13, k1a=0.8 * 3.95e-17, k1b=0.2 * 3.95e-17, k2a=1.2e-16,
                 k2b=1.2e-16, k3a=1.2e-17, k3b=1.0e-17, k4=1.1e-16, k5=2.0e-16, k6=0.2 * 3.0e-17)
        self.k = {m: v / rate for m, v in k.items()}
        Ei = rho * cs * cs / ((g - 1) * n)
        q = dict(q0a=0.73, q0b=2.8, q1a=0.29, q1b=0.84, q2a=4.3, q2b=0.81, q3a=0.42, q3b=1.16, q4=1.23, q5=1.81,
                 q6=0.42)
        self.q = {m: v * e / Ei for m, v in q.items()}
        self.tp = t_pulse * kg * cs
        self.photon = F0 / t_pulse / (c_light * h * (c_light / lam) * n)
        self.imap = torch.from_numpy(dk.imap).to(self.dev).reshape(self.ny, self.nx)

    # planes [variable][y][x], ghosted along x (and y in 2D)
    def ghosted(self, u):
        g = GHOSTS
        gy = g if self.nd == 2 else 0
        U = torch.zeros(self.nv, self.ny + 2 * gy, self.nx + 2 * g, dtype=torch.float64, device=self.dev)
        inner = U[:, gy:gy + self.ny, g:g + self.nx]
        inner.copy_(u)
        for z in self.boundary:
            kind, d, face = z[:3]
            N = self.dims[d]
            # planes along d, of the interior range across it
            V = U[:, gy:gy + self.ny] if d == 0 else U[:, :, g:g + self.nx].movedim(1, 2)
            for j in range(g):
                dst = j if face == 1 else N + g + j
                src = 2 * g - 1 - j if face == 1 else N + g - 1 - j
                if kind == "periodic":
                    src = dst + N if face == 1 else dst - N
                s = V[..., src]
                if kind in ("periodic", "extrapolate"):
                    V[..., dst] = s
                    continue
                G = self.zone_gamma
                rho, vx, vy = s[0], s[1] / s[0], s[2] / s[0]
                p = (s[3] - 0.5 * rho * (vx * vx + vy * vy)) * (G - 1)
                if kind == "supersonic-inflow":
                    rho, vx, vy, p = (torch.full_like(rho, v) for v in z[7:11])
                    for m in range(4, self.nv):
                        V[m, :, dst] = z[11 + m - 4]
                elif kind == "noslip-wall":
                    vx, vy = 2 * z[7] - vx, 2 * z[8] - vy
                elif kind != "supersonic-outflow":
                    raise ValueError(kind)
                V[0, :, dst], V[1, :, dst], V[2, :, dst] = rho, rho * vx, rho * vy
                V[3, :, dst] = p / (G - 1) + 0.5 * rho * (vx * vx + vy * vy)
        return U

    def prim(self, q):
        """velocities, pressure of [variable]... states"""
        v = [q[1 + i] / q[0] for i in range(self.nf - 2)]
        ke = sum(x * x for x in v)
        return v, (q[self.nf - 1] - 0.5 * q[0] * ke) * (self.gamma - 1)

    def flux(self, q, d):
        v, p = self.prim(q)
        f = q * v[d]
        f[1 + d] += p
        f[self.nf - 1] += p * v[d]
        return f

    def roe(self, a, b):
        """Roe average of two states: density, velocities, sound speed."""
        g = self.gamma
        (va, pa), (vb, pb) = self.prim(a), self.prim(b)
        ta, tb = a[0].sqrt(), b[0].sqrt()
        mix = lambda x, y: (ta * x + tb * y) / (ta + tb)  # noqa: E731
        v = [mix(x, y) for x, y in zip(va, vb)]
        H = mix(0.5 * sum(x * x for x in va) + g * pa / a[0] / (g - 1), 0.5 * sum(x * x for x in vb)
                + g * pb / b[0] / (g - 1))
        return ta * tb, v, ((g - 1) * (H - 0.5 * sum(x * x for x in v))).sqrt()

    def eig(self, rho, v, a, d):
        """Eigenvalues and left and right flow eigenvectors along d: acoustic
        fields, entropy field and, in 2D, the shear field."""
        g1 = self.gamma - 1
        un, ek = v[d], 0.5 * sum(x * x for x in v)
        one, zero = torch.ones_like(un), torch.zeros_like(un)
        if self.nf == 3:
            k = g1 / (rho * a)
            L = [[k * rho * (-ek + a * a / g1) / a, k * rho * un / a, -k * rho / a],
                 [k * (-ek - a * un / g1), k * (un + a / g1), -k],
                 [k * (ek - a * un / g1), k * (-un + a / g1), k]]
            h = a * a / g1 + ek
            c = rho / (2 * a)
            R = [[one, -c, c], [un, -c * (un - a), c * (un + a)], [ek, -c * (h - a * un), c * (h + a * un)]]
            return [un, un - a, un + a], L, R
        n = [1.0 if i == d else 0.0 for i in range(2)]
        aa, h = a * a, a * a / g1 + ek

        def acoustic(s):
            return [(g1 * ek - s * a * un) / (2 * aa)] + [(-g1 * v[i] + s * a * n[i]) / (2 * aa) for i in (0, 1)] + [
                g1 / (2 * aa)]

        entropy = [(aa - g1 * ek) / aa, g1 * v[0] / aa, g1 * v[1] / aa, -g1 / aa]
        t = 1 - d  # tangential; the shear field keeps the orientation (n_y, -n_x)
        sign = 1.0 if d == 1 else -1.0
        shear = [-sign * v[t], sign * one if t == 0 else zero, sign * one if t == 1 else zero, zero]
        L = [acoustic(-1.0), acoustic(1.0), shear, entropy]
        Rv = lambda s: [one, v[0] + s * a * n[0], v[1] + s * a * n[1], h + s * a * un]  # noqa: E731
        rs = [zero, sign * one if t == 0 else zero, sign * one if t == 1 else zero, sign * v[t]]
        cols = [Rv(-1.0), Rv(1.0), rs, [one, v[0], v[1], ek]]
        R = [[cols[j][i] for j in range(4)] for i in range(4)]
        return [un - a, un + a, un, un], L, R

    def times(self, M, x):
        return [sum(m * y for m, y in zip(row, x)) for row in M]

    def interfaces(self, q, f, d):
        """uL, uR, fL, fR of lines q, f [variable][line][N + 2 g] along d."""
        if not self.char:
            return [_line_values(s, left, self.crweno, self.kind) for s in (q, f) for left in (True, False)]
        n = q.shape[-1] - 2 * GHOSTS + 1
        _, L, R = self.eig(*self.roe(q[..., 2:2 + n], q[..., 3:3 + n]), d)
        out = []
        for s in (q, f):
            c = [self.times(L, s[:self.nf, :, k:k + n]) for k in range(6)]
            for left in (True, False):
                order = range(5) if left else range(5, 0, -1)
                w = [_weno5(self.kind, *[c[k][i] for k in order]) for i in range(self.nf)]
                o = torch.empty(self.nv, s.shape[1], n, dtype=torch.float64, device=self.dev)
                for i, x in enumerate(self.times(R, w)):
                    o[i] = x
                if self.nv > self.nf:
                    o[self.nf:] = _weno5(self.kind, *_stencil(s[self.nf:], left))
                out.append(o)
        return out

    def upwind(self, q, uL, uR, fL, fR, d):
        n = uL.shape[-1]
        nf = self.nf
        if self.upw == "roe":
            D, L, R = self.eig(*self.roe(q[..., 2:2 + n], q[..., 3:3 + n]), d)
            if nf == 4:  # Harten's entropy fix
                fix = lambda x: torch.where(x.abs() < 1e-6, (x * x + 1e-12) / 2e-6, x.abs())  # noqa: E731
            else:
                fix = torch.abs
            jump = 0.5 * (uR - uL)
            c = [fix(x) * y for x, y in zip(D, self.times(L, jump[:nf]))]
            f = 0.5 * (fL + fR)
            for i, x in enumerate(self.times(R, c)):
                f[i] -= x
            f[nf:] -= fix(D[0] if nf == 3 else D[3]) * jump[nf:]
            return f
        # rf-char: upwind by the sign of each eigenvalue at both interface states
        # and their Roe average, else local Lax-Friedrichs
        mean = self.roe(uL, uR)
        D, L, R = self.eig(*mean, d)

        def values(u):
            v, p = self.prim(u)
            a = (self.gamma * p / u[0]).sqrt()
            return [v[d] - a, v[d] + a, v[d], v[d]]

        eL, eR = values(uL), values(uR)

        def pick(i, ul, ur, fl, fr):
            lo, mid, hi = eL[i], D[i], eR[i]
            alpha = torch.maximum(torch.maximum(lo.abs(), mid.abs()), hi.abs())
            llf = 0.5 * (fl + fr + alpha * (ul - ur))
            plus = (lo > 0) & (mid > 0) & (hi > 0)
            minus = (lo < 0) & (mid < 0) & (hi < 0)
            return torch.where(plus, fl, torch.where(minus, fr, llf))

        parts = [self.times(L, x[:nf]) for x in (uL, uR, fL, fR)]
        c = [pick(i, *[x[i] for x in parts]) for i in range(nf)]
        f = pick(3, uL, uR, fL, fR)
        for i, x in enumerate(self.times(R, c)):
            f[i] = x
        return f

    def lines(self, U, d):
        """Lines of the ghosted planes along d, interior lines only."""
        g = GHOSTS
        if self.nd == 1:
            return U
        return U[:, g:-g] if d == 0 else U[:, :, g:-g].movedim(1, 2).contiguous()

    def d4(self, f):
        """Fourth-order difference along the last dimension, one-sided at the
        two outermost points of each side."""
        o = torch.empty_like(f)
        F = lambda k: f[..., k]  # noqa: E731
        o[..., 2:-2] = f[..., :-4] - 8 * f[..., 1:-3] + 8 * f[..., 3:-1] - f[..., 4:]
        o[..., 0] = -25 * F(0) + 48 * F(1) - 36 * F(2) + 16 * F(3) - 3 * F(4)
        o[..., 1] = -3 * F(0) - 10 * F(1) + 18 * F(2) - 6 * F(3) + F(4)
        o[..., -2] = -F(-5) + 6 * F(-4) - 18 * F(-3) + 10 * F(-2) + 3 * F(-1)
        o[..., -1] = 3 * F(-5) - 16 * F(-4) + 36 * F(-3) - 48 * F(-2) + 25 * F(-1)
        return o / 12

    def derivative(self, f, d):
        """d4 along d on the interior lines of ghosted planes, zero elsewhere."""
        g = GHOSTS
        o = torch.zeros_like(f)
        if d == 0:
            o[:, g:-g] = self.d4(f[:, g:-g])
        else:
            o[:, :, g:-g] = self.d4(f[:, :, g:-g].movedim(1, 2)).movedim(2, 1)
        return o

    def viscous(self, U):
        g = GHOSTS
        v, p = self.prim(U)
        T = self.gamma * p / U[0]
        P = torch.stack([v[0], v[1], T])
        ix, iy = self.inv[0][None, :], self.inv[1][:, None]
        X, Y = self.derivative(P, 0) * ix, self.derivative(P, 1) * iy
        Td = T * self.Tref
        r = torch.exp(1.5 * torch.log(Td / 275.0))
        mu = r * (275.0 + 110.4) / (Td + 110.4) / self.Re
        kap = r * (275.0 + 245.4 * math.exp(-27.6 / 275.0)) / (Td + 245.4 * torch.exp(-27.6 / Td))
        kap = kap / self.Re / (self.gamma - 1) / self.Pr
        txx, tyy = 2.0 / 3.0 * mu * (2 * X[0] - Y[1]), 2.0 / 3.0 * mu * (2 * Y[1] - X[0])
        txy = mu * (Y[0] + X[1])
        FX = torch.stack([txx, txy, v[0] * txx + v[1] * txy + kap * X[2]])
        FY = torch.stack([txy, tyy, v[0] * txy + v[1] * tyy + kap * Y[2]])
        par = self.derivative(FX, 0) * ix + self.derivative(FY, 1) * iy
        return par[:, g:-g, g:-g]

    def source(self, u, t):
        s = torch.zeros_like(u)
        k, q = self.k, self.q
        w = self.tp / 2.35482
        nh = self.imap * (self.photon * math.exp(-(t - self.tp) ** 2 / (2 * w * w)) if t > 0 else 0.0)
        O2, O3, D1, Dg, Su, Sg, CO2 = u[4:11]
        r0, r1, r2, r3 = nh * O3, D1 * O2, D1 * O3, O3 * Sg
        r4, r5, r6 = D1 * CO2, O3 * Su, Dg * O3
        s[5] = (-(k["k0a"] + k["k0b"]) * r0 - (k["k2a"] + k["k2b"]) * r2 - (k["k3a"] + k["k3b"]) * r3
                - k["k5"] * r5 - k["k6"] * r6)
        s[6] = k["k0a"] * r0 - (k["k1a"] + k["k1b"]) * r1 - (k["k2a"] + k["k2b"]) * r2 - k["k4"] * r4
        s[7] = k["k0a"] * r0 + k["k5"] * r5 - k["k6"] * r6
        s[8] = k["k2a"] * r2 - k["k5"] * r5
        s[9] = k["k1a"] * r1 - (k["k3a"] + k["k3b"]) * r3
        pair = lambda i: q["q%da" % i] * k["k%da" % i] + q["q%db" % i] * k["k%db" % i]  # noqa: E731
        s[3] = (pair(0) * r0 + pair(1) * r1 + pair(2) * r2 + pair(3) * r3 + q["q4"] * k["k4"] * r4
                + q["q5"] * k["k5"] * r5 + q["q6"] * k["k6"] * r6) / (self.gamma - 1)
        return s

    def rhs(self, u, t):
        U = self.ghosted(u)
        r = torch.zeros_like(u)
        for d in range(self.nd):
            q = self.lines(U, d)
            f = self.flux(q, d)
            fI = self.upwind(q, *self.interfaces(q, f, d), d)
            div = (fI[..., 1:] - fI[..., :-1]) * self.inv[d][GHOSTS:-GHOSTS]
            r -= div if d == 0 else div.movedim(1, 2)
        if self.nd == 2 and self.Re > 0:
            r[1:4] += self.viscous(U)
        if self.chem:
            r += self.source(u, t)
        return r

    def step(self, u, t):
        A, b = {"44": ([[0.5], [0, 0.5], [0, 0, 1.0]], [1 / 6, 1 / 3, 1 / 3, 1 / 6]),
                "ssprk3": ([[1.0], [0.25, 0.25]], [1 / 6, 1 / 6, 2 / 3])}[self.rk]
        k = [self.rhs(u, t)]
        for row in A:
            k.append(self.rhs(u + sum(self.dt * a * x for a, x in zip(row, k) if a), t + sum(row) * self.dt))
        return u + sum(self.dt * w * x for w, x in zip(b, k))

    def planes(self, u):
        return torch.from_numpy(np.ascontiguousarray(u)).to(self.dev).reshape(self.ny, self.nx, self.nv).movedim(
            2, 0).contiguous()

    def points(self, u):
        return u.movedim(0, 2).reshape(-1, self.nv).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        return None  # twenty members, minutes in plain torch
    if kind == "solve" and case["nx"] * case["ny"] > 3e6:
        return None  # over 20 seconds
    dk = _deck(case, seed)
    P = _Plain(dk)
    u = P.planes(dk.u)
    if kind == "rhs":
        return P.points(P.rhs(u, 0.45))
    if kind == "operators":
        U = P.ghosted(u)
        g = GHOSTS
        out = {"u": U.movedim(0, 2)}
        for d in (0, 1):
            out["f%d" % d] = P.flux(U, d).movedim(0, 2)
            # zero-filled corners have no flux (0/0 is taken as 0)
            out["f%d" % d] = torch.nan_to_num(out["f%d" % d], nan=0.0)
            q = P.lines(U, d)
            I = P.interfaces(q, P.flux(q, d), d)
            I.append(P.upwind(q, *I, d))
            for name, x in zip(("uL", "uR", "fL", "fR", "fI"), I):
                out["%s%d" % (name, d)] = x.permute(1, 2, 0) if d == 0 else x.permute(2, 1, 0)
            out["du%d" % d] = P.derivative(U, d).movedim(0, 2)
        return {k: v.contiguous() for k, v in out.items()}
    t = 0.0
    for _ in range(case["steps"]):
        u = P.step(u, t)
        t += P.dt
    return P.points(u)
