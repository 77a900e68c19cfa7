"""Assemblies into a kernel that the context holds already: another geometry of the
same shape, other shapes, another precision; bit-identical to a fresh context's."""
import numpy as np
import pytest

from unicycle_amd import PREC_F64, PREC_MIXED, configs

pytestmark = pytest.mark.gpu


def _set(eng, nx, nz, vn, seed):
    fault = configs.thrust_fault(nx=nx, nz=nz, ellipse=None)
    eng.set_elastic(fault.lambda_, fault.mu)
    eng.set_rectangles(*fault.geometry())
    eng.set_friction(*fault.friction())
    if vn:
        vol = configs.volume_grid(*vn, size=4000.0 + 100.0 * seed, top=20e3, origin=(0.0, 0.0))
        eng.set_volumes(*vol.geometry())
        eng.set_rheology(*vol.rheology())


@pytest.mark.parametrize("second", [(6, 3, (3, 3, 2), 1), (3, 6, (3, 3, 2), 2),
                                    (5, 3, (2, 2, 2), 3), (12, 6, (3, 3, 2), 4)])
@pytest.mark.parametrize("precision", [PREC_F64, PREC_MIXED])
def test_rebuild(engine_factory, second, precision):
    eng = engine_factory()
    _set(eng, 6, 3, (3, 3, 2), 0)
    eng.buildG(precision)
    first = eng.get_kernel()
    _set(eng, *second)
    eng.buildG(PREC_F64)
    fresh = engine_factory()
    _set(fresh, *second)
    fresh.buildG(PREC_F64)
    assert np.array_equal(eng.get_kernel(), fresh.get_kernel())
    _set(eng, 6, 3, (3, 3, 2), 0)
    eng.buildG(precision)
    assert np.array_equal(eng.get_kernel(), first)
