"""Ensemble states between the caller's layout and the groups', the attempts that a
run issues, and the shallow k-splits that small ensembles take."""
import numpy as np
import pytest

import orc
from unicycle_amd import PREC_BF16_I8, PREC_F64, PREC_SPLIT_BF16, configs
from unicycle_amd.ensemble import Ensemble

pytestmark = pytest.mark.gpu


def _ensemble(eng, precision, sizes, n_inst, seed=3):
    ens = Ensemble(eng, precision)
    rng = np.random.default_rng(seed)
    y0s = []
    for nx, nz in sizes:
        m = configs.thrust_fault(nx=nx, nz=nz, ellipse=None)
        d = configs.ensemble_instances(m, n_inst, seed=seed)
        y = rng.uniform(0.1, 1.0, (n_inst, m.n, 7))
        y[:, :, 5], y[:, :, 6] = 7.0 + 0.1 * y[:, :, 5], -9.0 + 0.01 * y[:, :, 6]
        y[:, :, 2:4] *= 60.0
        y0s.append((m, y.reshape(n_inst, -1)))
        ens.add_group(m, d["a"], d["b"], d["sig"], d["L"], y0s[-1][1])
    ens.build()
    return ens, y0s


# 7, 8, 9 elements: the tile of 8; 70 and 256 instances: several groups of 64
@pytest.mark.parametrize("nx,nz", [(1, 1), (7, 1), (4, 2), (3, 3), (11, 3)])
@pytest.mark.parametrize("n_inst", [1, 5, 64, 70, 256])
def test_reset_gives_the_initial_states(engine_factory, nx, nz, n_inst):
    eng = engine_factory()
    ens, y0s = _ensemble(eng, PREC_F64, [(nx, nz)], n_inst)
    for _ in range(2):
        got = np.concatenate([ens.state(g)[0] for g in range(len(ens.groups))])
        assert np.array_equal(got, y0s[0][1])
        st = ens.run(1e30, max_attempts=37, max_step=10.0)
        # no attempt is issued that no instance has left
        assert st.replays == 37 and st.attempts == 37 * n_inst
        for g in range(len(ens.groups)):
            y, t, dt, steps, att = ens.state(g)
            assert np.all(att == 37) and np.all(t > 0) and np.all(steps <= att)
        assert st.steps == sum(int(ens.state(g)[3].sum()) for g in range(len(ens.groups)))
        ens.reset()
    assert np.all(ens.state(0)[1] == 0.0) and np.all(ens.state(0)[4] == 0)
    ens.close()
    eng.close()


def test_two_groups_and_a_continued_run(engine_factory):
    eng = engine_factory()
    ens, y0s = _ensemble(eng, PREC_SPLIT_BF16, [(5, 3), (9, 4)], 6)
    for g in range(2):
        assert np.array_equal(ens.state(g)[0], y0s[g][1])
    whole = ens.run(1e30, max_attempts=50, max_step=10.0)
    end = [ens.state(g)[0] for g in range(2)]
    ens.reset()
    replays = 0
    for cap in (1, 20, 50):
        replays += ens.run(1e30, max_attempts=cap, max_step=10.0).replays
    assert replays == whole.replays == 50
    for g in range(2):
        assert np.array_equal(ens.state(g)[0], end[g])
    ens.close()
    eng.close()


@pytest.mark.parametrize("nx,nz", [(17, 9), (24, 12), (13, 3)])
@pytest.mark.parametrize("precision,bound", [(PREC_F64, 1e-14), (PREC_BF16_I8, 2.0 ** -13)])
def test_shallow_splits(engine_factory, nx, nz, precision, bound):
    """Every depth from 2 k-blocks per split up, remainders included, against
    binary64 (the bounds of the ensemble matvec)."""
    eng = engine_factory()
    ens, y0s = _ensemble(eng, precision, [(nx, nz)], 9)
    m = y0s[0][0]
    K = orc.buildG(orc.Mesh(m.lambda_, m.mu, rect=m.geometry()), nthreads=8)
    V = np.random.default_rng(1).standard_normal((2 * m.n, 9))
    want, scale = K @ V, np.abs(K) @ np.abs(V)
    nkb = (2 * m.n + 15) // 16
    for kb in [ens.tuning()[0], 2, 3, 4, 6, 8, 12, 16, 24]:
        if (nkb + kb - 1) // kb > 16:
            continue
        ens.set_tiling(kb, 0 if precision == PREC_F64 else 5)
        assert np.all(np.abs(ens.matvec(0, V) - want) <= bound * scale), kb
    ens.close()
    eng.close()


@pytest.mark.parametrize("precision", [PREC_F64, PREC_BF16_I8])
def test_equal_splits_are_timed_once(engine_factory, precision):
    """Depths that split K alike are one launch and share one timing: a build times
    each launch once, whatever the number of depths."""
    eng = engine_factory()
    for nx, nz in ((8, 4), (24, 12)):
        ens, y0s = _ensemble(eng, precision, [(nx, nz)], 8)
        nkb = -(-2 * y0s[0][0].n // 16)
        table = ens.tuning()[2].reshape(-1, 11)
        splits = [-(-nkb // kb) for kb in (32, 48, 64, 80, 96, 104, 128, 160, 192, 256, 512)]
        assert np.any(table > 0)
        for row in table:
            for s in set(splits):
                assert len({t for t, k in zip(row, splits) if k == s}) == 1
        ens.close()
    eng.close()
