"""Triangle columns of K in tiles of 64 receivers by 4 or 16 sources: sizes at
the edges of the tiles, patch and volume receivers, against the CPU oracle."""
import numpy as np
import pytest

import orc
from unicycle_amd import configs

pytestmark = pytest.mark.gpu


def _mesh(n):
    """The first n triangles of a curved, jittered mesh."""
    m = configs.megathrust_mesh(nx=28, ny=14, length=56e3, width=28e3, seed=5)
    return (m.i1[:n], m.i2[:n], m.i3[:n], m.vertices), m


def _close(K, want):
    # both differentiate the displacement exactly; the oracle's bound
    for c in range(3):
        a, b = K[c::3], want[c::3]
        assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b)


# 725: the first size in tiles of 16 sources with remainders in both directions
@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 130, 725])
def test_patch_receivers(engine_factory, n):
    tri, m = _mesh(n)
    eng = engine_factory()
    eng.set_elastic(m.lambda_, m.mu)
    eng.set_triangles(*tri)
    eng.buildG()
    _close(eng.get_kernel(), orc.buildG(orc.Mesh(m.lambda_, m.mu, tri=tri), nthreads=8))
    eng.close()


@pytest.mark.parametrize("n,nv", [(5, 1), (65, 12), (33, 70)])
def test_volume_receivers(engine_factory, n, nv):
    tri, m = _mesh(n)
    v = configs.volume_grid(nx=7, ny=5, nz=2, top=60e3)
    vol = tuple(np.ascontiguousarray(a[:nv]) for a in v.geometry())
    eng = engine_factory()
    eng.set_elastic(m.lambda_, m.mu)
    eng.set_triangles(*tri)
    eng.set_volumes(*vol)
    eng.buildG()
    K = eng.get_kernel()
    want = orc.buildG(orc.Mesh(m.lambda_, m.mu, tri=tri, vol=vol), nthreads=8)
    _close(K[:3 * n, :2 * n], want[:3 * n, :2 * n])
    # 60 to 75 km from triangles of 2 km: the twelve angular terms of a pair,
    # each of the size 1/r, cancel to L^2/r^3, so ten roundings of each (2.2e-16)
    # leave 12 * 10 * 2.2e-16 * (75/2)^2 = 3.7e-11 of the entries
    a, b = K[3 * n:, :2 * n], want[3 * n:, :2 * n]
    assert np.linalg.norm(a - b) <= 3.7e-11 * np.linalg.norm(b)
    eng.close()
