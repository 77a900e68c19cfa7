"""Ensemble states between the caller's layout and the groups', the attempts that a
run issues, and the shallow k-splits that small ensembles take."""
import numpy as np
import pytest

from unicycle_amd import PREC_F64, PREC_SPLIT_BF16, configs
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
