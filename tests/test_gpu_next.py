"""Steps whose assembly writes the next stage's state, the new solution and the
copied ghost points: solutions against the oracle over the Runge-Kutta tableaux
(two to four stages, with and without chemistry, whose stages have buffers of
their own) and the faces (copied by the kernel, or by the kernel after it), at
the edges of the 32 x 32 tiles.  Tolerance as for the other short solves: 1e-11
relative L2 of each variable."""
import numpy as np
import pytest

import _oracle as orc
import piafs_amd
from piafs_amd import decks

pytestmark = pytest.mark.gpu

TOL = 1e-11


def _face(kind, d, f, *vals, lo=-1e99, hi=1e99):
    return (kind, d, f, *((0, 0, lo, hi) if d == 0 else (lo, hi, 0, 0)), *vals)


FACES = {
    "periodic": [_face("periodic", d, f) for d in (0, 1) for f in (1, -1)],
    "mirror": [_face("extrapolate", d, f) for d in (0, 1) for f in (1, -1)],
    "mixed": [_face("periodic", 0, 1), _face("periodic", 0, -1), _face("extrapolate", 1, 1), _face("extrapolate", 1, -1)],
    "walls": [_face("extrapolate", d, f) for d in (0, 1) for f in (1, -1)]
    + [_face("noslip-wall", 1, 1, 0.1, 0.0), _face("slip-wall", 0, -1, 0.0, 0.0)],
    # a later zone that covers part of a face
    "part": [_face("extrapolate", d, f) for d in (0, 1) for f in (1, -1)] + [_face("slip-wall", 0, 1, 0.0, 0.0, lo=0.2, hi=0.5)],
}


def _check(tmp_path, dk, calls=(1, 3)):
    d = dk.write(str(tmp_path))
    o = orc.OCase(d)
    with piafs_amd.Case(d) as c:
        for n in calls:
            c.step(n)
            o.step(n)
            got, want = c.solution(), o.solution()
            assert np.all(np.isfinite(want))
            assert np.all(decks.rel_l2_per_var(got, want) <= TOL)
            c.rhs(dk.u, 0.1)  # uses the stage state; the next call starts from the solution


@pytest.mark.parametrize("nx,ny", [(31, 33), (32, 64), (35, 34), (65, 8)])
@pytest.mark.parametrize("faces", sorted(FACES))
@pytest.mark.parametrize("chem", [False, True])
def test_faces(tmp_path, nx, ny, faces, chem):
    _check(tmp_path, decks.ns2d_open_box(nx=nx, ny=ny, n_iter=10, boundary=FACES[faces], include_chemistry=chem, Re=500.0,
                                         flow=(1.0, 0.1, -0.05, None)))


@pytest.mark.parametrize("rk", ["1fe", "22", "33", "44", "ssprk3"])
@pytest.mark.parametrize("faces", ["periodic", "walls"])
@pytest.mark.parametrize("chem", [False, True])
def test_tableaux(tmp_path, rk, faces, chem):
    _check(tmp_path, decks.ns2d_open_box(nx=40, ny=33, n_iter=10, boundary=FACES[faces], include_chemistry=chem, rk=rk,
                                         Re=500.0, flow=(1.0, 0.1, -0.05, None)))


def test_layers_of_species(tmp_path):
    dk = decks.ns2d_photochem(nx=33, ny=31, n_iter=10, z_mm=3.0, rk="ssprk3")
    dk.u[:, 5::7] *= 1.0 + 0.1 * np.random.default_rng(3).uniform(-1, 1, dk.u[:, 5::7].shape)
    _check(tmp_path, dk)


def test_members_of_many_kinds(tmp_path):
    """1D members, single-stage ones and different tableaux in one batch equal their solo runs."""
    mem = [decks.ns2d_open_box(nx=40, ny=33, boundary=FACES[f], include_chemistry=ch, rk=rk, Re=500.0)
           for f, ch, rk in (("periodic", True, "44"), ("walls", True, "ssprk3"), ("mirror", False, "22"),
                             ("mixed", False, "1fe"))] + [decks.sod_1d(N=90)]
    dirs = [dk.write(str(tmp_path / str(k))) for k, dk in enumerate(mem)]
    solo = []
    for d in dirs:
        with piafs_amd.Case(d) as c:
            c.step(5)
            solo.append(c.solution())
    with piafs_amd.Batch(dirs) as b:
        b.step(2)
        b.step(3)
        for k in b.slots:
            assert np.array_equal(b.solution(k), solo[k]), k
