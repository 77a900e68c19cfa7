"""The resident integrator's plan (unicycle_amd/csrc/resident_plan.h) on the host.

Its exchange needs every block to publish slip rates: a plan has no block without
an element.  The sweep covers the three models, fault alone, volumes alone and
both, with either width of K's entries, around the sizes where the number of
blocks reaches the elements' and the largest number of blocks.
"""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "unicycle_amd",
                    "csrc")
SOURCE = """
#include "resident_plan.h"
extern "C" int plan(int model, int np, int nv, long m, long n, int f64, int cus, int *bounds, long *size)
{
    const ucy::ResidentPlan p = ucy::resident_plan(model, np, nv, m, n, f64, cus);
    if (!p.P) return 0;
    for (size_t i = 0; i < p.bounds.size(); i++) bounds[i] = p.bounds[i];
    const long s[] = {(long)p.bounds.size(), p.el_max, p.rows_max, p.rows_lds, p.rows_cached,
                      (long)p.lds};
    for (int i = 0; i < 6; i++) size[i] = s[i];
    return p.P;
}
"""
# rows and columns of K and state entries per patch and per volume
ROWS = {0: (3, 6), 1: (1, 2), 2: (2, 3)}
COLS = {0: (2, 6), 1: (1, 2), 2: (1, 3)}
STATE = {0: (7, 12), 1: (4, 4), 2: (6, 6)}
LDS = 158 * 1024


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, str(d / "plan.cpp"),
                    "-o", str(d / "plan.so")], check=True)
    f = ctypes.CDLL(str(d / "plan.so")).plan
    f.argtypes = [ctypes.c_int] * 3 + [ctypes.c_long] * 2 + [ctypes.c_int, ctypes.c_int,
                                                              ctypes.POINTER(ctypes.c_int),
                                                              ctypes.POINTER(ctypes.c_long)]

    def call(model, np_, nv, f64, cus=256):
        m = ROWS[model][0] * np_ + ROWS[model][1] * nv
        n = COLS[model][0] * np_ + COLS[model][1] * nv
        n += n & 1
        bounds, size = (ctypes.c_int * 300)(), (ctypes.c_long * 6)()
        P = f(model, np_, nv, m, n, f64, cus, bounds, size)
        return m, n, P, list(bounds[:P + 1]), list(size)
    return call


def _check(plan, model, np_, nv, f64, cus=256):
    m, n, P, b, (count, el, rows, lds_rows, cached, lds) = plan(model, np_, nv, f64, cus)
    if not P:
        return False
    what = (model, np_, nv, f64, cus)
    assert P <= min(cus, 256) and count == P + 1 and b[0] == 0 and b[-1] == np_ + nv, what
    assert all(x < y for x, y in zip(b, b[1:])), (what, "a block without an element")
    rp, rv = ROWS[model]
    first = [rp * min(e, np_) + rv * max(e - np_, 0) for e in b]
    assert max(y - x for x, y in zip(b, b[1:])) <= el <= 64 and el % 2 == 0, what
    assert max(y - x for x, y in zip(first, first[1:])) <= rows and rows % 2 == 0, what
    state = STATE[model][1 if nv else 0]
    entry = 8 if f64 else 4
    assert 0 <= lds_rows <= rows and cached >= lds_rows, what
    assert lds == 8 * (n + 2 * state * el + 2 * rows) + lds_rows * n * entry <= LDS, what
    return True


@pytest.mark.parametrize("f64", [True, False], ids=["f64", "reduced"])
@pytest.mark.parametrize("model", [0, 1, 2], ids=["3d", "antiplane", "planestrain"])
def test_every_block_has_an_element(plan, model, f64):
    rng = np.random.default_rng(model)
    sizes = [(1, 0), (0, 1), (2, 0), (0, 2), (39, 200), (390, 50), (36, 168), (91, 100), (13, 3)]
    sizes += [(i, 0) for i in range(3, 1500, 7)] + [(0, i) for i in range(3, 1500, 7)]
    sizes += [(int(a), int(b)) for a, b in np.exp(rng.uniform(0.0, np.log(2500.0), (1500, 2)))]
    planned = sum(_check(plan, model, np_, nv, f64) for np_, nv in sizes)
    assert planned > len(sizes) // 2


@pytest.mark.parametrize("cus", [1, 32, 64, 304])
def test_at_most_a_block_per_cu(plan, cus):
    """A device partition has fewer CUs; more elements than its blocks take are
    left to the captured attempt."""
    for f64 in (True, False):
        planned = [_check(plan, 0, np_, nv, f64, cus)
                   for np_, nv in [(20, 0), (390, 0), (945, 0), (39, 200), (2048, 0), (4096, 0)]]
        assert planned == [n <= 64 * cus for n in (20, 390, 945, 239, 2048, 4096)]


def test_limits(plan):
    """K beyond its limit, or more elements than the blocks take, is left to the
    captured attempt; a K that fits one block takes one."""
    assert plan(0, 4096, 0, True)[2] == 256 and plan(0, 4800, 0, True)[2] == 0
    assert plan(0, 8192, 0, False)[2] == 256 and plan(0, 10000, 0, False)[2] == 0
    assert plan(1, 56, 0, True)[2] == 1 and plan(1, 57, 0, True)[2] == 2
    assert plan(0, 45, 0, True)[2] == 1 and plan(0, 46, 0, True)[2] == 3
