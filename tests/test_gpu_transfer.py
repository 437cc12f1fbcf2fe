"""States crossing between host and device in chunks: what goes in comes out,
bit for bit, at the edges of the chunking (one chunk, chunks of unequal size,
more chunks than buffers)."""
import threading

import numpy as np
import pytest

import piafs_amd
from piafs_amd import decks

pytestmark = pytest.mark.gpu


# 88 B a point: 17 x 13 one short chunk; 149 x 10 just over, 1489 x 1 at 24 B
# far below one chunk (128 KiB); 301 x 257 eight uneven chunks; 701 x 463 and
# its neighbour more than eight chunks of 2 MiB
@pytest.mark.parametrize("nx,ny", [(17, 13), (149, 10), (301, 257), (701, 463), (464, 703)])
def test_state_round_trip(tmp_path, nx, ny):
    dk = decks.ns2d_photochem(nx=nx, ny=ny, n_iter=1)
    r = np.random.default_rng(nx * 1000 + ny)
    u = r.standard_normal(dk.u.shape)
    with piafs_amd.Case(dk.write(str(tmp_path))) as c:
        assert np.array_equal(c.solution(), dk.u)
        c.set_solution(u)
        assert np.array_equal(c.solution(), u)
        v = r.standard_normal(dk.u.shape)  # buffers still in use by the first upload are waited for
        c.set_solution(u)
        c.set_solution(v)
        assert np.array_equal(c.solution(), v)


def test_state_round_trip_1d_and_threads(tmp_path):
    """Two cases of different sizes on two threads share one device's buffers."""
    out = {}

    def work(name, dk):
        u = np.random.default_rng(7).standard_normal(dk.u.shape)
        with piafs_amd.Case(dk.write(str(tmp_path / name))) as c:
            ok = True
            for _ in range(5):
                c.set_solution(u)
                ok = ok and np.array_equal(c.solution(), u)
                u = u[::-1].copy()
            out[name] = ok

    ts = [threading.Thread(target=work, args=a) for a in
          (("line", decks.sod_1d(N=1489, n_iter=1)), ("grid", decks.ns2d_photochem(nx=401, ny=203, n_iter=1)))]
    for d in ("line", "grid"):
        (tmp_path / d).mkdir()
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert out == {"line": True, "grid": True}
