"""The CRWENO5 line systems over segment lengths and team widths: right-hand
sides against the oracle on lines that fill a team exactly, by one row less and
one more, in both sweeps, paired (Roe) and split (llf-char), and every
reconstruction alone through the device-buffer operator.  Tolerance as for the
other pieces of a right-hand side: 1e-12 of each variable's largest magnitude."""
import numpy as np
import pytest

import _oracle as orc
import piafs_amd
from piafs_amd import decks

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _close(got, want):
    got, want = got.reshape(-1, got.shape[-1]), want.reshape(-1, want.shape[-1])
    scale = np.abs(want).max(axis=0)
    assert np.all(np.abs(got - want).max(axis=0) <= TOL * np.where(scale > 0, scale, 1.0))


def _deck(nx, ny, **kw):
    periodic = [("periodic", 0, 1, 0, 0, -1e99, 1e99), ("periodic", 0, -1, 0, 0, -1e99, 1e99),
                ("periodic", 1, 1, -1e99, 1e99, 0, 0), ("periodic", 1, -1, -1e99, 1e99, 0, 0)]
    return decks.ns2d_open_box(nx=nx, ny=ny, flow=(1.0, 0.3, -0.2, None), scheme="crweno5", include_chemistry=True,
                               Re=500.0, boundary=periodic, **kw)


# interior rows N - 1 at, below and above 4, 6, .. 16 rows on 1 .. 256 lanes
SIZES = [(5, 8), (9, 17), (33, 34), (64, 66), (97, 98), (129, 130), (161, 12), (193, 194), (225, 14), (257, 256),
         (321, 10), (449, 9), (577, 8), (641, 7), (769, 8), (898, 7), (1024, 8), (1025, 6), (1026, 6), (1281, 7),
         (1537, 6), (2049, 5), (4097, 5), (6, 1500)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("upwinding", ["roe", "llf-char"])
def test_segment_lengths(tmp_path, nx, ny, upwinding):
    dk = _deck(nx, ny, upwinding=upwinding)
    u = dk.u * (1.0 + 1e-2 * np.random.default_rng(nx + ny).uniform(-1, 1, dk.u.shape))
    d = dk.write(str(tmp_path))
    want = orc.OCase(d).rhs(u, 0.45)
    with piafs_amd.Case(d) as c:
        _close(c.rhs(u, 0.45), want)


@pytest.mark.parametrize("rows", [4, 6, 8, 10, 12, 14, 16])
@pytest.mark.parametrize("weights", ["js", "mapped", "z", "yc", "none"])
def test_rows_and_weights(tmp_path, rows, weights):
    """Lines of 8 lanes of each segment length, the last one a row short."""
    dk = _deck(8 * rows, 8 * rows, weights=weights)
    u = dk.u * (1.0 + 1e-2 * np.random.default_rng(rows).uniform(-1, 1, dk.u.shape))
    d = dk.write(str(tmp_path))
    want = orc.OCase(d).rhs(u, 0.45)
    with piafs_amd.Case(d) as c:
        _close(c.rhs(u, 0.45), want)


def test_members_of_many_shapes(tmp_path):
    """Members share the choice of segment lengths; each equals its solo run."""
    dirs = []
    for k, (nx, ny) in enumerate([(33, 97), (129, 65), (200, 40), (1100, 9), (50, 300), (257, 31)]):
        dirs.append(_deck(nx, ny, n_iter=2, dt=1e-4).write(str(tmp_path / str(k))))
    with piafs_amd.Batch(dirs) as b:
        b.step(2)
        got = [b.solution(k) for k in b.slots]
    for k, d in enumerate(dirs):
        with piafs_amd.Case(d) as c:
            c.step(2)
            assert np.array_equal(got[k], c.solution()), k


# from 2^15 cells on the species' cell fluxes are formed in the line teams: narrow
# and wide teams, one sweep of each, and the first sizes on either side; the last
# has teams of 128 lanes whose pairs write the species' interface fluxes
@pytest.mark.parametrize("nx,ny", [(182, 181), (181, 181), (1100, 33), (31, 1100), (1026, 259)])
@pytest.mark.parametrize("upwinding", ["roe", "rf-char"])
def test_species_fluxes_in_the_teams(tmp_path, nx, ny, upwinding):
    dk = _deck(nx, ny, upwinding=upwinding)
    r = np.random.default_rng(nx)
    u = dk.u * (1.0 + 1e-2 * r.uniform(-1, 1, dk.u.shape))
    u[:, 6:] = 1e-3 * r.uniform(0.5, 1.0, u[:, 6:].shape)
    d = dk.write(str(tmp_path))
    want = orc.OCase(d).rhs(u, 0.45)
    with piafs_amd.Case(d) as c:
        _close(c.rhs(u, 0.45), want)


def test_autotuning_tries_the_choice_by_size(tmp_path):
    """Lines of 896 and 448 rows fill teams of 14 rows a lane, which is not among
    the uniform candidates, where 16 rows a lane would leave an eighth idle:
    tuning keeps them."""
    d = _deck(897, 449, n_iter=2).write(str(tmp_path))
    with piafs_amd.Case(d) as c:
        rows, ms = c.autotune()
        c.profile(True)
        c.step(1)
        c.sync()
        assert "recon_14" in c.kernel_times()
    assert rows == 16 and ms > 0.0


# the segment length chosen for each of these lines, on 32 to 64, 128 and 256
# lanes, the last one a row short
@pytest.mark.parametrize("n,across,cls", [(128, 9, "4"), (384, 9, "6"), (512, 9, "8"), (640, 9, "10"), (768, 9, "12"),
                                          (896, 9, "14"), (1024, 9, "16"), (1280, 9, "w10"), (1536, 17, "w12"),
                                          (2048, 33, "w16"), (2560, 5, "w10"), (3072, 5, "w12"), (4096, 5, "w16")])
@pytest.mark.parametrize("weights", ["js", "mapped", "z", "yc", "none"])
def test_every_variant_with_every_weight(tmp_path, n, across, cls, weights):
    nx, ny = (n, across) if weights in ("js", "z", "none") else (across, n)
    dk = _deck(nx, ny, weights=weights, n_iter=1, dt=1e-5)
    u = dk.u * (1.0 + 1e-2 * np.random.default_rng(n).uniform(-1, 1, dk.u.shape))
    d = dk.write(str(tmp_path))
    want = orc.OCase(d).rhs(u, 0.45)
    with piafs_amd.Case(d) as c:
        _close(c.rhs(u, 0.45), want)
        c.profile(True)
        c.step(1)
        c.sync()
        assert "recon_" + cls in c.kernel_times()
