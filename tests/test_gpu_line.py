"""1D cases advanced by whole steps (one launch for many steps, or one a step):
the same bits with timing marks around the launches, from the kernels of a
stage, which lines beside a 2D member take, and the oracle's values."""
import numpy as np
import pytest

import _oracle as orc
import piafs_amd
from piafs_amd import decks

pytestmark = pytest.mark.gpu

# the reflect rule negates every variable, density too: those runs turn to NaN,
# and have to do so at the same points
ENDS = {
    "mirror": None,
    "periodic": [("periodic", 0, 1, 0, 0), ("periodic", 0, -1, 0, 0)],
    "walls": [("slip-wall", 0, 1, 0, 0, 0.1), ("slip-wall", 0, -1, 0, 0, -0.2)],
    "reflect": [("reflect", 0, 1, 0, 0), ("extrapolate", 0, -1, 0, 0)],
}


def _same(tmp_path, dk, steps, finite=True):
    d = dk.write(str(tmp_path))
    with piafs_amd.Case(d) as a, piafs_amd.Case(d) as b:
        b.profile(True)
        for n in steps:
            a.step(n)
            b.step(n)
            a.sync()
            b.sync()
            got, want = a.solution(), b.solution()
            assert np.all(np.isfinite(want)) or not finite
            assert np.array_equal(got, want, equal_nan=True)


def _deck(N, ends, scheme, interp, upwinding, rk, weights=0):
    dk = decks.sod_1d(N=N, scheme=scheme, interp=interp, upwinding=upwinding, rk=rk, boundary=ENDS[ends], mapped=weights)
    r = np.random.default_rng(N)
    dk.u[:, 0] *= 1.0 + 0.02 * r.uniform(-1, 1, N)
    dk.u[:, 1] = 0.1 * dk.u[:, 0]
    return dk


# windows that keep 51 (RK3), 45 (RK4) points: less than one, exactly, one more, many
@pytest.mark.parametrize("N", [8, 45, 51, 52, 90, 300])
@pytest.mark.parametrize("ends", sorted(ENDS))
@pytest.mark.parametrize("interp,upwinding,rk", [("characteristic", "roe", "ssprk3"), ("components", "rf-char", "44"),
                                                 ("characteristic", "llf-char", "44"), ("components", "rusanov", "1fe")])
def test_windows(tmp_path, N, ends, interp, upwinding, rk):
    _same(tmp_path, _deck(N, ends, "weno5", interp, upwinding, rk), (1, 4, 3), ends != "reflect")


# teams of 4 and 8 rows a lane, full and not, the last and first size of each;
# 514 goes the general way on both sides
@pytest.mark.parametrize("N", [8, 33, 128, 257, 258, 513, 514])
@pytest.mark.parametrize("ends,upwinding", [("mirror", "roe"), ("periodic", "rf-char"), ("walls", "llf-char"),
                                            ("reflect", "rusanov")])
def test_line_systems(tmp_path, N, ends, upwinding):
    _same(tmp_path, _deck(N, ends, "crweno5", "components", upwinding, "44", weights=N & 1), (1, 6), ends != "reflect")


def test_members_together(tmp_path):
    """Lines of both kinds in a batch, and with a 2D member, equal their solo runs."""
    mem = [_deck(70, "mirror", "weno5", "characteristic", "roe", "ssprk3"),
           _deck(129, "periodic", "crweno5", "components", "roe", "44"),
           _deck(300, "walls", "crweno5", "components", "roe", "44"),
           _deck(111, "periodic", "weno5", "components", "roe", "44")]
    two = decks.ns2d_photochem(nx=20, ny=12, n_iter=5)
    dirs = [dk.write(str(tmp_path / str(k))) for k, dk in enumerate(mem + [two])]
    solo = []
    for d in dirs:
        with piafs_amd.Case(d) as c:
            c.step(5)
            solo.append(c.solution())
    for some in (dirs[:4], dirs):
        with piafs_amd.Batch(some) as b:
            b.step(2)
            b.step(3)
            for k in b.slots:
                assert np.array_equal(b.solution(k), solo[k]), k


@pytest.mark.parametrize("scheme,interp", [("weno5", "characteristic"), ("crweno5", "components")])
def test_no_steps(tmp_path, scheme, interp):
    """Step counts of zero and less leave the solution and the time as they are,
    before the first step and after an odd and an even number of them."""
    d = _deck(90, "mirror", scheme, interp, "roe", "44").write(str(tmp_path))
    with piafs_amd.Case(d) as c:
        for n in (0, 1, 1):
            c.step(n)
            u, t = c.solution(), c.info.t
            for none in (0, -1, -2):
                c.step(none)
                assert np.array_equal(c.solution(), u), none
                assert c.info.t == t


@pytest.mark.parametrize("N,scheme,interp,names", [(128, "crweno5", "components", {"line_4"}),
                                                   (300, "crweno5", "components", {"line_8"}),
                                                   (90, "weno5", "characteristic", {"tube", "tube_back"})])
def test_profiled_steps_are_the_steps(tmp_path, N, scheme, interp, names):
    """A profiled case takes the launches that it takes otherwise."""
    with piafs_amd.Case(_deck(N, "mirror", scheme, interp, "roe", "44").write(str(tmp_path))) as c:
        c.profile(True)
        c.step(3)
        c.sync()
        times = c.kernel_times()
    assert set(times) == names and all(t > 0.0 for t in times.values())


def _beside_2d(tmp_path, decks_1d, steps, finite=True):
    """Lines that step together with a 2D member go through the kernels of a
    stage: alone they give the same bits."""
    dirs = [dk.write(str(tmp_path / str(k))) for k, dk in enumerate(decks_1d)]
    two = decks.ns2d_photochem(nx=20, ny=12, n_iter=sum(steps)).write(str(tmp_path / "two"))
    with piafs_amd.Batch(dirs + [two]) as b:
        for n in steps:
            b.step(n)
        want = [b.solution(k) for k in b.slots[:-1]]
    for d, w, dk in zip(dirs, want, decks_1d):
        with piafs_amd.Case(d) as c:
            for n in steps:
                c.step(n)
            assert np.all(np.isfinite(w)) or not finite, dk.u.shape
            assert np.array_equal(c.solution(), w, equal_nan=True), dk.u.shape


@pytest.mark.parametrize("ends", sorted(ENDS))
@pytest.mark.parametrize("interp,upwinding,rk", [("characteristic", "roe", "ssprk3"), ("components", "rf-char", "44"),
                                                 ("characteristic", "llf-char", "44"), ("components", "rusanov", "1fe")])
def test_windows_against_stage_kernels(tmp_path, ends, interp, upwinding, rk):
    mem = [_deck(N, ends, "weno5", interp, upwinding, rk) for N in (8, 45, 51, 52, 90, 300)]
    _beside_2d(tmp_path, mem, (1, 4, 3), ends != "reflect")


@pytest.mark.parametrize("ends,upwinding", [("mirror", "roe"), ("periodic", "rf-char"), ("walls", "llf-char"),
                                            ("reflect", "rusanov")])
def test_line_systems_against_stage_kernels(tmp_path, ends, upwinding):
    mem = [_deck(N, ends, "crweno5", "components", upwinding, "44", weights=N & 1) for N in (8, 33, 128, 257, 258, 513)]
    _beside_2d(tmp_path, mem, (1, 6), ends != "reflect")


def _scheme(dk, weights):
    dk.weno.update(mapped=0, borges=int(weights == "z"), yc=int(weights == "yc"), no_limiting=int(weights == "none"))
    return dk


@pytest.mark.parametrize("weights", ["z", "yc", "none"])
def test_other_weights(tmp_path, weights):
    """Every weight rule is a kernel of its own: both kinds of lines, and upw5."""
    mem = [_scheme(_deck(N, "mirror", *how, "44"), weights)
           for N, how in [(61, ("weno5", "characteristic", "roe")), (62, ("weno5", "components", "rf-char")),
                          (63, ("upw5", "components", "roe")), (64, ("upw5", "characteristic", "llf-char")),
                          (100, ("crweno5", "components", "roe")), (300, ("crweno5", "components", "rf-char"))]]
    _beside_2d(tmp_path, mem, (1, 5))


@pytest.mark.parametrize("scheme,interp,weights", [("weno5", "characteristic", "z"), ("weno5", "components", "yc"),
                                                   ("weno5", "components", "none"), ("upw5", "components", "none"),
                                                   ("crweno5", "components", "z"), ("crweno5", "components", "yc"),
                                                   ("crweno5", "components", "none")])
def test_weights_against_the_oracle(tmp_path, scheme, interp, weights):
    """10 steps; relative L2 norm of the difference per variable, the bound of the
    other parity tests."""
    dk = _scheme(_deck(100, "periodic", scheme, interp, "roe", "44"), weights)
    dk.u[:] = dk.u[0] * (1.0 + 0.05 * np.sin(2 * np.pi * np.arange(100)[:, None] / 100))
    d = dk.write(str(tmp_path))
    o = orc.OCase(d)
    o.step(10)
    with piafs_amd.Case(d) as c:
        c.step(10)
        assert np.all(decks.rel_l2_per_var(c.solution(), o.solution()) <= 1e-11)
