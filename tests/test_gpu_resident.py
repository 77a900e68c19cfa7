"""The resident integrator (one kernel for many attempts) against the captured
attempt (a graph of kernels per attempt).

Both call the same element functions and sum each row in the same order, so a
run has to give the same bits on either: state, times, step lengths, maxima,
error ratios, rejections and observed entries.  A run that also logs an
observation point's displacement takes the captured attempt; without it, a
kernel of this size takes the resident one.

Sizes: one element; the largest models of one block (56 segments, 45 patches) and
the next ones, of two and three; blocks' shares that
do not divide; rows that do not fit the blocks' LDS; every model, with volumes;
the reduced forms of K; a run split into calls; an end time, a step limit and a
run that ends in an error; observed entries; two runs at once; the hand-over to the
captured attempt at the start, between launches and after a wait that ran out.
"""
import threading

import numpy as np
import pytest

from unicycle_amd import PREC_F64, PREC_MIXED, PREC_SPLIT_BF16, UcyError, configs

pytestmark = pytest.mark.gpu

HUGE = 1.0e30


def _segments(make, n):
    eng = make()
    w = np.full(n, 400.0)
    x = np.zeros((n, 3))
    x[:, 2] = 400.0 * np.arange(n)
    one = np.ones(n)
    z = (np.arange(n) + 0.5) / n
    b = np.where((z > 0.2) & (z < 0.8), 0.014, 0.006)
    eng.set_antiplane(30e3, x, w, np.full(n, np.pi / 2))
    eng.set_friction(1e-9 * one, 0 * one, 0.6 * one, 100.0 * one, 0.010 * one, b, 0.01 * one,
                     1e-6 * one, 5.0 * one)
    return eng


def _thrust(make, nx, nz):
    m = configs.thrust_fault(nx=nx, nz=nz, ellipse=None)
    eng = make()
    eng.set_elastic(m.lambda_, m.mu)
    eng.set_rectangles(*m.geometry())
    eng.set_friction(*m.friction())
    return eng


def _volumes(make, nx, nz, v):
    eng = _thrust(make, nx, nz)
    g = configs.volume_grid(nx=v[0], ny=v[1], nz=v[2], top=60e3)
    eng.set_volumes(*g.geometry())
    eng.set_rheology(*g.rheology())
    return eng


def _antiplane_volumes(make, n, n2, n3):
    m = configs.antiplane_viscous(n, n2, n3)
    f = m.fault
    eng = make()
    eng.set_antiplane(f.mu, f.x, f.width, f.dip)
    eng.set_antiplane_volumes(m.vx, m.thickness, m.vwidth, m.vdip)
    eng.set_friction(*f.friction())
    eng.set_rheology(*m.rheology())
    return eng


def _planestrain(make, n, n2=0, n3=0):
    m = configs.planestrain_viscous(n, n2, n3) if n2 else None
    f = m.fault if m else configs.planestrain_fault(n)
    eng = make()
    eng.set_planestrain(f.lambda_, f.mu, f.x, f.width, f.dip)
    if m:
        eng.set_planestrain_volumes(m.vx, m.thickness, m.vwidth, m.vdip)
    eng.set_friction(*f.friction())
    if m:
        eng.set_rheology(*m.rheology())
    return eng


MODELS = {
    "antiplane-1": lambda mk: _segments(mk, 1),
    "antiplane-2": lambda mk: _segments(mk, 2),
    "antiplane-56": lambda mk: _segments(mk, 56),
    "antiplane-57": lambda mk: _segments(mk, 57),
    "antiplane-64": lambda mk: _segments(mk, 64),
    "antiplane-65": lambda mk: _segments(mk, 65),
    "antiplane-111": lambda mk: _segments(mk, 111),
    "antiplane-850": lambda mk: _segments(mk, 850),
    "thrust-1": lambda mk: _thrust(mk, 1, 1),
    "thrust-44": lambda mk: _thrust(mk, 11, 4),
    "thrust-45": lambda mk: _thrust(mk, 9, 5),
    "thrust-46": lambda mk: _thrust(mk, 23, 2),
    "thrust-247": lambda mk: _thrust(mk, 19, 13),
    "thrust-1081": lambda mk: _thrust(mk, 47, 23),
    "thrust-2816": lambda mk: _thrust(mk, 64, 44),
    "antiplane-volumes": lambda mk: _antiplane_volumes(mk, 41, 5, 7),
    "planestrain-51": lambda mk: _planestrain(mk, 51),
    "planestrain-volumes": lambda mk: _planestrain(mk, 24, 4, 3),
    "volumes": lambda mk: _volumes(mk, 7, 5, (3, 3, 2)),
    "volumes-large": lambda mk: _volumes(mk, 13, 7, (5, 5, 4)),
    # more blocks than a volume's rows allow at equal cuts: ranges without an
    # element are dropped from the plan
    "volumes-39-200": lambda mk: _volumes(mk, 13, 3, (10, 5, 4)),
    "volumes-390-50": lambda mk: _volumes(mk, 26, 15, (5, 5, 2)),
}


def _start(eng):
    y = eng.initStateVector()
    rng = np.random.default_rng(3)
    if eng.antiplane:
        y[3:4 * eng.np:4] += 0.01 * rng.standard_normal(eng.np)
    elif eng.planestrain:
        y[4:5 * eng.np:5] += 0.01 * rng.standard_normal(eng.np)
    else:
        y[6:7 * eng.np:7] += 0.01 * rng.standard_normal(eng.np)
        y[4:7 * eng.np:7] = rng.uniform(0.1, 1.0, eng.np)
    return y


def _same(a, b):
    assert (a.steps, a.attempts, a.rhs_evals) == (b.steps, b.attempts, b.rhs_evals)
    assert a.time == b.time and a.dt_next == b.dt_next and a.vmax == b.vmax
    for k in ("y", "t_log", "dt_log", "vmax_log", "errmax_log", "reject_log", "emax_log", "obs_y",
              "obs_dydt"):
        assert np.array_equal(getattr(a, k), getattr(b, k)), k


@pytest.mark.parametrize("name", MODELS)
def test_same_bits_as_the_captured_attempt(engine_factory, name):
    eng = MODELS[name](engine_factory)
    eng.buildG()
    y = _start(eng)
    eng.buildO(np.array([[1e3, 2e3, 0.0]]))
    obs = [0, y.size // 2, y.size - 1]
    kw = dict(max_steps=120, log_cap=120, history=True, observe=obs)
    _same(eng.integrate(y, HUGE, **kw), eng.integrate(y, HUGE, displacement=True, **kw))
    eng.close()


@pytest.mark.parametrize("name", ["thrust-45", "thrust-247", "volumes", "volumes-large",
                                  "volumes-39-200", "volumes-390-50"])
@pytest.mark.parametrize("precision", [PREC_MIXED, PREC_SPLIT_BF16])
def test_reduced_precision(engine_factory, name, precision):
    eng = MODELS[name](engine_factory)
    eng.buildG(precision)
    y = _start(eng)
    eng.buildO(np.array([[1e3, 2e3, 0.0]]))
    kw = dict(max_steps=60, log_cap=60, history=True, observe=[0, 3], max_step=1e6)
    _same(eng.integrate(y, HUGE, **kw), eng.integrate(y, HUGE, displacement=True, **kw))
    eng.close()


def test_largest(engine_factory):
    """No row fits LDS beside the slip rates."""
    eng = _thrust(engine_factory, 128, 64)
    eng.buildG(PREC_MIXED)
    y = _start(eng)
    eng.buildO(np.array([[1e3, 2e3, 0.0]]))
    kw = dict(max_steps=12, log_cap=12, history=True)
    a, b = eng.integrate(y, HUGE, **kw), eng.integrate(y, HUGE, displacement=True, **kw)
    assert np.array_equal(a.y, b.y) and np.array_equal(a.errmax_log, b.errmax_log)
    eng.close()


@pytest.mark.parametrize("n", [1, 111])
def test_a_run_in_pieces(engine_factory, n):
    eng = _segments(engine_factory, n)
    eng.buildG()
    y = _start(eng)
    whole = eng.integrate(y, HUGE, max_steps=90, log_cap=90)
    t, dt, times = 0.0, 1e-3, []
    for k in (1, 2, 40, 47):
        r = eng.integrate(y, HUGE, dt0=dt, max_steps=k, log_cap=k, t0=t)
        y, t, dt = r.y, r.time, r.dt_next
        times.append(r.t_log)
    assert np.array_equal(np.concatenate(times), whole.t_log)
    assert np.array_equal(y, whole.y)
    eng.close()


def test_more_attempts_than_one_launch_takes(engine_factory):
    """A launch ends after 2000 attempts at the latest, also between the
    rejected attempts of a step."""
    eng = _segments(engine_factory, 1)
    eng.set_kernel(np.array([[-7 * np.pi / 16 * 30e3 / 6e3]]))
    y = _start(eng)
    eng.buildO(np.array([[0.0, 1e3, 0.0]]))
    a = eng.integrate(y, HUGE, max_steps=4500, log_cap=4500, max_step=1e7, history=True)
    b = eng.integrate(y, HUGE, max_steps=4500, log_cap=4500, max_step=1e7, history=True,
                      displacement=True)
    assert a.attempts > 4000 and a.reject_log.sum() > 0
    assert np.array_equal(a.y, b.y) and np.array_equal(a.t_log, b.t_log)
    assert np.array_equal(a.reject_log, b.reject_log)
    eng.close()


def test_end_time_and_errors(engine_factory):
    eng = _thrust(engine_factory, 9, 5)
    eng.buildG()
    y = _start(eng)
    r = eng.integrate(y, 5.0e5, max_step=1e5, log_cap=100)
    assert r.time >= 5.0e5 and r.t_log[-2] < 5.0e5
    bad = y.copy()
    bad[6] = np.nan
    with pytest.raises(UcyError, match="non-finite"):
        eng.integrate(bad, HUGE, max_steps=5)
    again = eng.integrate(y, 5.0e5, max_step=1e5, log_cap=100)
    assert np.array_equal(again.y, r.y)
    eng.close()


@pytest.mark.parametrize("name", ["antiplane-1", "thrust-247", "volumes-large",
                                  "planestrain-volumes", "thrust-1081"])
def test_every_entry_observed(engine_factory, name):
    """All entries in a shuffled order, some of them three times, and at next to no
    cost: the time per attempt without observed entries, and half as much for the
    stores (measured: 6 % at most; 11 to 30 times when every lane looked through
    the whole list)."""
    eng = MODELS[name](engine_factory)
    eng.buildG()
    y = _start(eng)
    eng.buildO(np.array([[1e3, 2e3, 0.0]]))
    rng = np.random.default_rng(5)
    obs = rng.permutation(np.concatenate([np.arange(y.size), [0, 0, y.size - 1, y.size // 2]]))
    kw = dict(max_steps=60, log_cap=60, history=True)
    _same(eng.integrate(y, HUGE, observe=obs, **kw),
          eng.integrate(y, HUGE, observe=obs, displacement=True, **kw))
    few, many = (min(eng.integrate(y, HUGE, observe=o, **kw).wall_seconds for _ in range(5))
                 for o in ([0], obs))
    assert many < 1.5 * few + 1e-3
    eng.close()


# ---- the hand-over to the captured attempt ------------------------------------
def _handed_over(eng, y, launches, attempts, wait, kw):
    eng.set_resident_limits(launches, attempts, wait)
    r = eng.integrate(y, HUGE, **kw)
    info = eng.resident_info()
    eng.set_resident_limits()
    return r, info


@pytest.mark.parametrize("precision", [PREC_F64, PREC_MIXED, PREC_SPLIT_BF16])
@pytest.mark.parametrize("name", ["thrust-247", "volumes-39-200", "thrust-1081"])
def test_a_wait_that_runs_out(engine_factory, name, precision):
    """With no time to wait no block gets the others' first values: every block
    leaves at the end of its first attempt, and the call goes back to where the
    launch began."""
    eng = MODELS[name](engine_factory)
    eng.buildG(precision)
    y = _start(eng)
    kw = dict(max_steps=30, log_cap=30, history=True, observe=[0, y.size - 1], max_step=1e6)
    want = eng.integrate(y, HUGE, **kw)
    assert eng.resident_info()[0] >= 1 and eng.resident_info()[1] == 0
    got, info = _handed_over(eng, y, -1, 0, 0.0, kw)
    assert info == (0, 3)
    _same(got, want)
    _same(eng.integrate(y, HUGE, **kw), want)
    eng.close()


@pytest.mark.parametrize("precision", [PREC_F64, PREC_MIXED])
@pytest.mark.parametrize("launches", [0, 1, 2, 3, 7])
def test_no_room_after_some_launches(engine_factory, launches, precision):
    """One attempt per launch: the captured attempt goes on after a step, and
    after rejected attempts of a step."""
    eng = MODELS["thrust-247"](engine_factory)
    eng.buildG(precision)
    y = _start(eng)
    # the first step is rejected several times
    kw = dict(dt0=1e8, epsilon=1e-9, max_steps=20, log_cap=20, history=True, observe=[0, 5])
    want = eng.integrate(y, HUGE, **kw)
    assert want.reject_log[0] >= 2 and eng.resident_info()[1] == 0
    got, info = _handed_over(eng, y, launches, 1, -1.0, kw)
    assert info == (launches, 2)
    _same(got, want)
    eng.close()


@pytest.mark.parametrize("name", ["thrust-247", "thrust-1081", "volumes-39-200"])
def test_two_contexts_at_once(engine_factory, name):
    """Two runs share the device's CUs, or take turns at them (256 blocks of nearly
    all LDS, several launches each), or leave them for the captured attempt."""
    engs = [MODELS[name](engine_factory) for _ in range(2)]
    for e in engs:
        e.buildG()
    y = _start(engs[0])
    kw = dict(max_steps=300, log_cap=300, history=True, observe=[0, 3])
    for e in engs:
        e.set_resident_limits(attempts=40)
    want = engs[0].integrate(y, HUGE, **kw)
    got = [None, None]

    def run(i):
        got[i] = engs[i].integrate(y, HUGE, **kw)
    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in got:
        _same(g, want)
    for e in engs:
        e.close()
