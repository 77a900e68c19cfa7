"""Strain-volume sums: the reduced corner sums that every pair off the planes of a
volume's vertical faces takes, and the formula text that pairs on them keep.

Against the oracle (the formula text, differentiated in forward mode).  Its sums
round some 8 corners x 22 integrals x 8 terms, each a quotient that loses up to
(R2/s)^2 = 40 to 1 - (p/R2)^2 at these distances (s >= 3 km of R2 <= 19 km from a
corner's vertical line): 1408 x 40 x 1.1e-16 = 6e-12 of the largest term, so 1e-11
of the norm over sources that include near ones.
"""
import numpy as np
import pytest

import orc

pytestmark = pytest.mark.gpu


def _oracle(fn, nout, x, frame, src, eps, G, lam):
    y, L, T, W, st = src
    out = [np.zeros(L.size) for _ in range(nout)]
    getattr(orc.oracle(), fn)(
        orc.p(orc.f64(x)), *[orc.p(orc.f64(f)) for f in frame], L.size, orc.p(orc.f64(y)),
        orc.p(L), orc.p(T), orc.p(W), orc.p(st), orc.p(orc.f64(eps)), orc.D(G), orc.D(lam),
        *[orc.p(o) for o in out])
    return np.stack(out)


def _both(eng, x, frame, src, eps, G, lam):
    y, L, T, W, st = src
    for fn, name, n in ((eng.computeTractionKernelsVerticalStrainVolume,
                         "orc_traction_kernels_strainvolume", 3),
                        (eng.computeStressKernelsVerticalStrainVolume,
                         "orc_stress_kernels_strainvolume", 6)):
        yield (np.stack(fn(x, *frame, L.size, y, L, T, W, st, *eps, G, lam)),
               _oracle(name, n, x, frame, src, eps, G, lam))


def _frame(rng):
    q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    return q[:, 0], q[:, 1], q[:, 2]


@pytest.mark.parametrize("ns", [1, 63, 64, 65, 129])
@pytest.mark.parametrize("lam", [30e3, 0.0, 70e3, -15e3])
@pytest.mark.parametrize("where", ["deep", "surface", "top", "bottom", "inside"])
def test_matches_the_formula_text(engine_factory, ns, lam, where):
    """Receivers at the depths of a volume's top and bottom (the branch cuts of the
    angles), at the surface with a volume that reaches it, and inside one."""
    eng = engine_factory()
    rng = np.random.default_rng(ns)
    # corners at 2 km x odd or 1.5 km x odd, receivers at 0 and 250 m
    y = np.column_stack([4e3 * rng.integers(-2, 2, ns) + 2e3, 4e3 * rng.integers(-2, 2, ns),
                         1e3 * rng.integers(0, 12, ns)]).astype(float)
    L, T, W = np.full(ns, 4e3), np.full(ns, 4e3), rng.choice([1e3, 3e3], ns)
    y[0] = (-2e3, 0.0, 0.0 if where == "surface" else 5e3)
    W[0] = 3e3
    src = (y, L, T, W, np.zeros(ns))
    x = np.array([0.0, 250.0, {"deep": 13250.0, "surface": 0.0, "top": 5e3, "bottom": 8e3,
                               "inside": 6250.0}[where]])
    frame = _frame(rng)
    for j in range(6):
        eps = np.eye(6)[j]
        for got, want in _both(eng, x, frame, src, eps, 30e3, lam):
            assert np.isfinite(got).all()
            assert np.linalg.norm(got - want) <= 1e-11 * np.linalg.norm(want)


@pytest.mark.parametrize("x1,x2", [(0.0, 700.0), (4e3, 700.0), (-9e3, 2e3), (1e3, -2e3),
                                   (0.0, 0.0), (0.0, 2e3), (4e3, -2e3)])
@pytest.mark.parametrize("x3", [0.0, 5e3, 6e3])
def test_on_the_planes_of_the_faces(engine_factory, x1, x2, x3):
    """0/0 and infinities stand where the formula text has them, pair by pair: one
    volume has the receiver on its face's plane, its neighbours do not."""
    eng = engine_factory()
    y = np.array([[0.0, 0.0, 5e3], [-33e3, 1e3, 4e3], [7e3, 31e3, 1e3]])
    src = (y, np.full(3, 4e3), np.full(3, 4e3), np.full(3, 3e3), np.zeros(3))
    frame = _frame(np.random.default_rng(3))
    for j in range(6):
        eps = np.eye(6)[j]
        for got, want in _both(eng, np.array([x1, x2, x3]), frame, src, eps, 30e3, 30e3):
            assert np.array_equal(np.isnan(got), np.isnan(want))
            assert np.array_equal(np.isinf(got), np.isinf(want))
            # the neighbours, 8 sizes away: their sums are 1/500 of their terms, so
            # 100 times the other test's bound
            ok = np.isfinite(want)
            assert np.isfinite(want[:, 1:]).all()
            assert np.linalg.norm((got - want)[ok]) <= 1e-9 * np.linalg.norm(want[ok])


def test_incompressible_medium(engine_factory):
    """lambda beyond 2^53 G: nu is 1/2 and the stress factor infinite, in both."""
    eng = engine_factory()
    y = np.array([[0.0, 0.0, 5e3], [9e3, 1e3, 4e3]])
    src = (y, np.full(2, 4e3), np.full(2, 4e3), np.full(2, 3e3), np.full(2, 0.3))
    frame = _frame(np.random.default_rng(4))
    for j in range(6):
        for got, want in _both(eng, np.array([3e3, 700.0, 6e3]), frame, src, np.eye(6)[j], 1.0,
                               1e30):
            assert np.array_equal(np.isnan(got), np.isnan(want))
