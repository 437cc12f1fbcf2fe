"""bench.py's byte model of a launch follows the line teams the library takes."""
import sys

import pytest

from conftest import ROOT

sys.path.insert(0, ROOT)
import bench  # noqa: E402


# lanes = rows of a line / rows of a lane, to a power of two: 32 .. 128 write the
# species' fluxes
@pytest.mark.parametrize("n,kernel,fused", [(64, "recon_4", False), (128, "recon_4", True), (256, "recon_8", True),
                                            (256, "recon_16", False), (1024, "recon_16", True),
                                            (1100, "recon_w10", True), (1281, "recon_w10", True),
                                            (2049, "recon_w16", True), (2300, "recon_w10", False)])
def test_species_fluxes_follow_the_teams(n, kernel, fused):
    rows = bench.line_rows([kernel, "flux", "upwind", "recon_ends"])
    assert rows == int(kernel.split("_")[1].strip("w"))
    assert bench.species_fused(n, 11, True, rows) is fused
    assert not bench.species_fused(n, 11, False, rows) and not bench.species_fused(n, 4, True, rows)
    faces = n * (n + 1)
    assert bench.kernel_algorithmic_bytes("upwind", n, 11, 3, True, rows) == 16 * faces * (20 if fused else 41)


def test_velocity_plane_from_its_size_on():
    """1024 x 1024: 11 variables and 5 planes of fluxes in, 16 interface arrays out;
    below 2^15 cells all fluxes."""
    pos, faces = 1024 * 1030, 1024 * 1025
    assert bench.kernel_algorithmic_bytes("recon_16", 1024, 11, 3, True, 16) == 16 * (16 * pos + 16 * faces)
    assert bench.kernel_algorithmic_bytes("flux", 1024, 11, 3, True, 16) == 16 * (9 * pos + faces)
    assert bench.kernel_algorithmic_bytes("flux", 128, 11, 3, True, 4) == 16 * (22 * 128 * 134 + 128 * 129)
    assert bench.kernel_algorithmic_bytes("recon_ends", 128, 11, 3, True, 4) is None
