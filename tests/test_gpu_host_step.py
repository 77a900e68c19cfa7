"""A host's own step loop: odefun, RKCKm and RKQSm with one launch per stage.

RKCKm against its own definition, six odefun calls and the Cash-Karp sums on the
host: the sums are rounded alike (no fused operations on either side), the matvec
of a stage is the same device code, so solution and error are equal bit for bit.
Sizes at the edges of the launches: 1 element, 4 and 5 (a block's wavefronts), 64
and 65 (the first kernel's block), with and without volumes; the 2-D models, whose
elements have 4, 5 and 6 state entries."""
import numpy as np
import pytest

from unicycle_amd import PREC_F64, PREC_MIXED, PREC_SPLIT_BF16, configs

pytestmark = pytest.mark.gpu

A = {2: (0.2,), 3: (3.0 / 40.0, 9.0 / 40.0), 4: (0.3, -0.9, 1.2),
     5: (-11.0 / 54.0, 2.5, -70.0 / 27.0, 35.0 / 27.0),
     6: (1631.0 / 55296.0, 175.0 / 512.0, 575.0 / 13824.0, 44275.0 / 110592.0, 253.0 / 4096.0)}
C = {1: 37.0 / 378.0, 3: 250.0 / 621.0, 4: 125.0 / 594.0, 6: 512.0 / 1771.0}
DC = {1: C[1] - 2825.0 / 27648.0, 3: C[3] - 18575.0 / 48384.0, 4: C[4] - 13525.0 / 55296.0,
      5: -277.0 / 14336.0, 6: C[6] - 0.25}


def _thrust(eng, nx, nz, vol):
    fault = configs.thrust_fault(nx=nx, nz=nz, ellipse=None)
    eng.set_elastic(fault.lambda_, fault.mu)
    eng.set_rectangles(*fault.geometry())
    eng.set_friction(*fault.friction())
    if vol:
        v = configs.volume_grid(*vol, size=4000.0, top=20e3, origin=(0.0, 0.0))
        eng.set_volumes(*v.geometry())
        eng.set_rheology(*v.rheology())


def _plane(eng, model, n, vol):
    m = getattr(configs, model + "_viscous")(n, *vol) if vol else None
    f = m.fault if m else getattr(configs, model + "_fault")(n)
    if model == "antiplane":
        eng.set_antiplane(f.mu, f.x, f.width, f.dip)
    else:
        eng.set_planestrain(f.lambda_, f.mu, f.x, f.width, f.dip)
    if vol:
        getattr(eng, "set_" + model + "_volumes")(m.vx, m.thickness, m.vwidth, m.vdip)
    eng.set_friction(*f.friction())
    if vol:
        eng.set_rheology(*m.rheology())


@pytest.mark.parametrize("nx,nz,vol", [(1, 1, None), (4, 1, None), (5, 1, None), (8, 8, None),
                                       (13, 5, None), (3, 2, (2, 2, 1)), (13, 5, (5, 4, 3))])
@pytest.mark.parametrize("precision", [PREC_F64, PREC_MIXED, PREC_SPLIT_BF16])
def test_one_launch_per_stage(engine_factory, nx, nz, vol, precision):
    eng = engine_factory()
    _thrust(eng, nx, nz, vol)
    _check(eng, precision, vol)


@pytest.mark.parametrize("model", ["antiplane", "planestrain"])
@pytest.mark.parametrize("n,vol", [(1, None), (65, None), (24, (4, 3))])
@pytest.mark.parametrize("precision", [PREC_F64, PREC_MIXED])
def test_2d_models(engine_factory, model, n, vol, precision):
    eng = engine_factory()
    _plane(eng, model, n, vol)
    _check(eng, precision, vol)


def _check(eng, precision, vol):
    eng.buildG(precision)
    y = eng.initStateVector(1 if vol else 0)
    n = y.size
    rng = np.random.default_rng(n)
    y = y * (1.0 + 1e-3 * rng.uniform(-1.0, 1.0, n))
    k = {1: np.empty(n)}
    eng.odefun(n, 0.0, y, k[1])
    h = 1e3
    for s in range(2, 7):
        if s == 2:
            yt = y + (h * 0.2) * k[1]
        else:
            yr = A[s][0] * k[1]
            for j in range(1, s - 1):
                yr = yr + A[s][j] * k[j + 1]
            yt = y + h * yr
        k[s] = np.empty(n)
        eng.odefun(n, 0.0, yt, k[s])
    yr = C[1] * k[1]
    for j in (3, 4, 6):
        yr = yr + C[j] * k[j]
    yout, yerr = np.empty(n), np.empty(n)
    eng.RKCKm(n, 0.0, y, k[1], h, yout, yerr)
    assert np.array_equal(yout, y + h * yr)
    er = DC[1] * k[1]
    for j in (3, 4, 5, 6):
        er = er + DC[j] * k[j]
    assert np.array_equal(yerr, h * er)
    # RKQSm accepts this step under a loose bound and leaves it under a tight one
    ys, big = y.copy(), np.full(n, 1e30)
    t, hdid, _ = eng.RKQSm(n, 0.0, ys, k[1], big, h)
    assert (t, hdid) == (h, h) and np.array_equal(ys, yout)
    ys = y.copy()
    tight = np.maximum(np.abs(yerr), 1e-300) / 1e-6 / 20.0
    t, hdid, _ = eng.RKQSm(n, 0.0, ys, k[1], tight, h)
    assert 0.0 < hdid < h and not np.array_equal(ys, yout)
    # an integration on the same context in between does not disturb the buffers
    eng.integrate(y, 1e9, max_steps=3)
    again = np.empty(n)
    eng.RKCKm(n, 0.0, y, k[1], h, again, yerr)
    assert np.array_equal(again, yout)
