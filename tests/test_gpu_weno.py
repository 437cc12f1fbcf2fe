"""The schemes without line systems (WENO5, upw5): interface fluxes and the
right-hand side against the oracle, at the edges of the kernel's tiles of 64
interfaces and over the schemes, weights and upwinders it dispatches on.
Tolerance as for the other pieces of a right-hand side: 1e-12 of each
variable's largest magnitude."""
import numpy as np
import pytest

import _oracle as orc
import piafs_amd
from piafs_amd import decks

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _check(tmp_path, dk):
    r = np.random.default_rng(5)
    u = dk.u * (1.0 + 1e-3 * r.uniform(-1, 1, dk.u.shape))
    d = dk.write(str(tmp_path))
    ref = orc.OCase(d)
    P, rhs_ref = ref.rhs_parts(u, 0.45), ref.rhs(u, 0.45)
    with piafs_amd.Case(d) as c:
        fi = [c.interface_flux(u, 0.45, k) for k in range(dk.solver["ndims"])]
        rhs = c.rhs(u, 0.45)
    for got, want in [(f, P["fi%d" % k]) for k, f in enumerate(fi)] + [(rhs, rhs_ref)]:
        got, want = got.reshape(-1, got.shape[-1]), want.reshape(-1, want.shape[-1])
        scale = np.abs(want).max(axis=0)
        assert np.all(np.abs(got - want).max(axis=0) <= TOL * np.where(scale > 0, scale, 1.0))


# (N + 1) lines across a tile's end, exactly one tile, one interface more
@pytest.mark.parametrize("nx,ny", [(7, 9), (63, 6), (64, 7), (31, 127)])
@pytest.mark.parametrize("interp", ["components", "characteristic"])
@pytest.mark.parametrize("upwinding", ["roe", "rf-char", "llf-char", "rusanov"])
def test_tiles_and_upwinders(tmp_path, nx, ny, interp, upwinding):
    _check(tmp_path, decks.ns2d_open_box(nx=nx, ny=ny, flow=(1.0, 0.3, -0.2, None), interp=interp, upwinding=upwinding,
                                         include_chemistry=ny != 9, Re=500.0))


@pytest.mark.parametrize("weights", ["mapped", "z", "yc", "none"])
@pytest.mark.parametrize("interp", ["components", "characteristic"])
def test_weights(tmp_path, weights, interp):
    _check(tmp_path, decks.ns2d_open_box(nx=30, ny=21, flow=(1.0, 0.3, -0.2, None), interp=interp, weights=weights,
                                         include_chemistry=True, Re=500.0))


@pytest.mark.parametrize("upwinding", ["roe", "rf-char", "rusanov"])
@pytest.mark.parametrize("interp", ["components", "characteristic"])
def test_several_layers_of_species(tmp_path, interp, upwinding):
    """Three layers: more species than the kernel holds at a time."""
    dk = decks.ns2d_photochem(nx=20, ny=17, n_iter=1, scheme="weno5", interp=interp, upwinding=upwinding, z_mm=3.0)
    assert dk.u.shape[1] == 25
    rho = dk.u[:, 0]
    dk.u[:, 1], dk.u[:, 2] = 0.2 * rho, -0.1 * rho
    dk.u[:, 3] += 0.5 * 0.05 * rho
    _check(tmp_path, dk)


@pytest.mark.parametrize("N", [8, 63, 64, 200])
@pytest.mark.parametrize("interp", ["components", "characteristic"])
@pytest.mark.parametrize("upwinding", ["roe", "rf-char", "llf-char", "rusanov"])
def test_lines(tmp_path, N, interp, upwinding):
    dk = decks.sod_1d(N=N, interp=interp, upwinding=upwinding)
    dk.u[:, 1] = 0.3 * dk.u[:, 0]
    _check(tmp_path, dk)
