"""The work that users have this engine do, as measurable cases.

Each case is one call (or one short loop of calls) of the public entry points:

``segments``   the main loop of the 2-D antiplane programs and of the 0-D
               spring-slider (one segment): ``Engine.integrate`` with the step
               log that the programs write to time.txt;
``fault``      the main loop of the 3-D rate-and-state program on a dipping
               thrust of Okada rectangles or on a curved mesh of triangles, K in
               binary64, mixed or split bf16;
``host_step``  the loop of a Fortran host that keeps its own main loop and
               calls ``odefun`` and ``RKQSm`` on host arrays, step by step;
``rectangles``, ``triangles``, ``volumes``
               the assembly ``buildG`` of the three source types (the volume
               model with its fault, so all four blocks of K);
``ensemble``   a batched ensemble: reset to the initial states, a run of some
               attempts, and every group's state read back.

Results are given in the parts that they consist of (slip, traction, state
variable, slip rate, time), as these differ by many orders of magnitude.
``exact`` restates the physics in binary64 torch (Okada 1992, Nikkhoo and
Walter 2015, the aging law, Cash-Karp RK45 with RKQS).
"""
import math

import numpy as np
import torch

from unicycle_amd import (Engine, PREC_BF16_I8, PREC_F64, PREC_MIXED, PREC_SPLIT_BF16, configs)
from unicycle_amd.ensemble import Ensemble

PRECISION = {"f64": PREC_F64, "mixed": PREC_MIXED, "split_bf16": PREC_SPLIT_BF16,
             "bf16_i8": PREC_BF16_I8}
NEVER = 1.0e30        # an end time that no run here reaches
SHORT_STEP = 1.0e5    # s, the longest step of the ensembles and of reduced precision
# matrices up to this size can stay on the chip between the right-hand sides of
# one call; larger ones have to be read from memory for each of them
ON_CHIP = 128e6


def listed():
    return [
        # the 0-D spring-slider program: nothing but latency
        {"name": "spring_slider", "kind": "segments", "segments": 1, "steps": 400, "max_step": 1.0e7},
        # a 2-D antiplane fault of an odd number of segments
        {"name": "antiplane_241", "kind": "segments", "segments": 241, "steps": 200,
         "max_step": 1.0e7},
        # a small 3-D mesh of triangles, with steps of any length
        {"name": "mesh_390", "kind": "fault", "mesh": "triangles", "nx": 15, "nz": 13,
         "precision": "f64", "steps": 150, "max_step": 3.0e6},
        # the 64 x 32 thrust, the plain method's model
        {"name": "thrust_2048", "kind": "fault", "mesh": "rectangles", "nx": 64, "nz": 32,
         "precision": "f64", "steps": 120, "max_step": 3.0e6},
        # a large fault in the reduced precision that keeps a binary64 step start
        {"name": "thrust_8192_mixed", "kind": "fault", "mesh": "rectangles", "nx": 128, "nz": 64,
         "precision": "mixed", "steps": 40, "max_step": SHORT_STEP},
        # the drop-in Fortran host: its own loop over odefun and RKQSm
        {"name": "host_step_945", "kind": "host_step", "mesh": "rectangles", "nx": 35, "nz": 27,
         "steps": 20, "max_step": 3.0e6},
        # assembly of the three source types
        {"name": "assemble_2048_rectangles", "kind": "rectangles", "nx": 64, "nz": 32,
         "precision": "f64"},
        {"name": "assemble_2952_triangles", "kind": "triangles", "nx": 41, "ny": 36},
        {"name": "assemble_fault_volumes", "kind": "volumes", "nx": 18, "nz": 13, "vx": 11,
         "vy": 9, "vz": 6},
        # the uneven ensemble, 4 geometries x 64 instances
        {"name": "ensemble_mixed_sizes", "kind": "ensemble",
         "groups": "32x32,64x32,64x64,128x64", "instances": 64, "precision": "bf16_i8",
         "attempts": 60},
        # one 4096-patch geometry, 256 instances sharing its K
        {"name": "ensemble_256_shared", "kind": "ensemble", "groups": "64x64", "instances": 256,
         "precision": "bf16_i8", "attempts": 60},
        # a small ensemble of odd sizes in binary64
        {"name": "ensemble_odd_f64", "kind": "ensemble", "groups": "24x12,17x9", "instances": 37,
         "precision": "f64", "attempts": 60},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["segments", "segments", "fault", "fault", "fault", "host_step",
                       "rectangles", "triangles", "volumes", "ensemble", "ensemble"])
    if kind == "segments":
        n = _log_int(rng, 30, 900) if rng.random() < 0.85 else 1
        return {"kind": kind, "segments": n, "steps": rng.randint(30, 250), "max_step": 1.0e7}
    if kind == "fault":
        precision = rng.choice(["f64", "f64", "f64", "mixed", "split_bf16"])
        mesh = rng.choice(["rectangles", "triangles"])
        most = (96, 48) if mesh == "rectangles" else (40, 24)
        return {"kind": kind, "mesh": mesh, "nx": _log_int(rng, 4, most[0]),
                "nz": _log_int(rng, 3, most[1]), "precision": precision,
                "steps": rng.randint(20, 40), "max_step": 3.0e6 if precision == "f64" else SHORT_STEP}
    if kind == "host_step":
        return {"kind": kind, "mesh": "rectangles", "nx": _log_int(rng, 4, 64),
                "nz": _log_int(rng, 3, 32), "steps": rng.randint(5, 20), "max_step": 3.0e6}
    if kind == "rectangles":
        return {"kind": kind, "nx": _log_int(rng, 5, 64), "nz": _log_int(rng, 5, 48),
                "precision": rng.choice(["f64", "f64", "mixed"])}
    if kind == "triangles":
        return {"kind": kind, "nx": _log_int(rng, 3, 41), "ny": _log_int(rng, 3, 36)}
    if kind == "volumes":
        return {"kind": kind, "nx": _log_int(rng, 3, 18), "nz": _log_int(rng, 2, 13),
                "vx": _log_int(rng, 2, 11), "vy": _log_int(rng, 2, 9), "vz": _log_int(rng, 1, 6)}
    n = rng.randint(1, 3)
    groups = ",".join("%dx%d" % (_log_int(rng, 8, 80), _log_int(rng, 6, 40)) for _ in range(n))
    instances = _log_int(rng, 3, 256 if n == 1 else 64)
    return {"kind": kind, "groups": groups, "instances": instances,
            "precision": rng.choice(["bf16_i8", "bf16_i8", "split_bf16", "mixed", "f64"]),
            "attempts": rng.randint(20, 40)}


# ---- the models -----------------------------------------------------------

def _thrust(nx, nz, seed):
    """A thrust whose patch size, dip and depth come from the seed."""
    rng = np.random.default_rng(seed)
    return configs.thrust_fault(nx=nx, nz=nz, patch=float(rng.uniform(1500.0, 2500.0)),
                                dip_deg=float(rng.uniform(15.0, 50.0)),
                                top=float(rng.uniform(300.0, 3000.0)), ellipse=None)


def _accumulated(y, rake, rng):
    """The slip and normal traction of a run under way.  (From zero they enter
    the error norm relative to their own first increments, where one rounding
    of an entry near a sign change sets the length of the steps.)"""
    slip = rng.uniform(0.5, 1.0, y.shape[:-1])
    y[..., 0], y[..., 1] = slip * np.cos(rake), slip * np.sin(rake)
    y[..., 4] = rng.uniform(0.2, 1.0, y.shape[:-1])


def _instances(model, count, seed):
    """Per-instance friction and the states of a run under way: the reference's
    initial tractions, a perturbed slip rate, the state variable at steady
    state."""
    d = configs.ensemble_instances(model, count, seed=seed)
    rng = np.random.default_rng(seed + 1)
    y = np.zeros((count, model.n, 7))
    tau = d["sig"] * (model.mu0 + (d["a"] - d["b"]) * np.log(model.Vpl / model.Vo)) \
        - model.damping * model.Vpl
    V = model.Vpl * (1.0 + 1e-3 * rng.standard_normal((count, model.n)))
    y[:, :, 2], y[:, :, 3] = tau * np.cos(model.rake), tau * np.sin(model.rake)
    y[:, :, 5], y[:, :, 6] = np.log10(d["L"] / V), np.log10(V)
    _accumulated(y, model.rake, rng)
    return d, y.reshape(count, -1)


def _segments(case, seed):
    """Vertical segments of 500 m (one: the point source of the 0-D program)
    and their friction; the slip rate is perturbed about the plate rate."""
    n = case["segments"]
    rng = np.random.default_rng(seed)
    # the point source's radius is large enough for stick-slip
    width = float(rng.uniform(300.0, 600.0)) if n > 1 else float(rng.uniform(5e3, 8e3))
    x = np.zeros((n, 3))
    x[:, 2] = width * np.arange(n)
    one = np.ones(n)
    z = (np.arange(n) + 0.5) / n
    a = 0.010 * one
    b = np.where((z > 0.2) & (z < 0.7), 0.014, 0.006) if n > 1 else 0.014 * one
    mu, L = 30e3, float(rng.uniform(0.01, 0.02))
    fric = (1e-9 * one, 0.0 * one, 0.6 * one, float(rng.uniform(50.0, 150.0)) * one, a, b,
            L * one, 1e-6 * one, 5.0 * one)
    V = 1e-9 * (1.0 + (1e-2 * rng.standard_normal(n) if n > 1 else rng.uniform(0.2, 0.5, 1)))
    y = np.zeros((n, 4))
    y[:, 1] = fric[3] * (0.6 + (a - b) * math.log(1e-3)) - 5.0 * 1e-9
    y[:, 2], y[:, 3] = np.log10(L / V), np.log10(V)
    return mu, x, width * one, fric, y.reshape(-1)


def _spring(mu, width):
    return np.array([[-7.0 * math.pi / 16.0 * mu / width[0]]])


def _volume_model(case, seed):
    rng = np.random.default_rng(seed)
    fault = _thrust(case["nx"], case["nz"], seed)
    vol = configs.volume_grid(nx=case["vx"], ny=case["vy"], nz=case["vz"],
                              size=float(rng.uniform(3000.0, 5000.0)),
                              top=float(rng.uniform(60e3, 70e3)),
                              origin=(float(rng.uniform(-2e4, 2e4)), float(rng.uniform(-4e4, 0.0))))
    return fault, vol


def _mesh(nx, ny, seed):
    return configs.megathrust_mesh(nx=nx, ny=ny, length=2e3 * nx, width=1e3 * ny, seed=seed)


def _fault(case, seed):
    """Geometry, friction and initial state of one 3-D fault."""
    if case["mesh"] == "rectangles":
        m = _thrust(case["nx"], case["nz"], seed)
        d, y = _instances(m, 1, seed)
        return m, configs.instance_friction(m, d, 0), y[0]
    m = _mesh(case["nx"], case["nz"], seed)
    Vpl, rake, mu0, sig, a, b, L, Vo, damping = m.friction()
    tau = sig * (mu0 + (a - b) * np.log(Vpl / Vo)) - damping * Vpl
    rng = np.random.default_rng(seed + 1)
    V = Vpl * (1.0 + 1e-2 * rng.standard_normal(m.n))
    y = np.zeros((m.n, 7))
    y[:, 2], y[:, 3] = tau * np.cos(rake), tau * np.sin(rake)
    y[:, 5], y[:, 6] = np.log10(L / V), np.log10(V)
    _accumulated(y, rake, rng)
    return m, m.friction(), y.reshape(-1)


def _groups(case):
    return [tuple(int(v) for v in g.split("x")) for g in case["groups"].split(",")]


# ---- prepare and run ------------------------------------------------------

def _engine(lambda_, mu):
    eng = Engine(0)
    eng.set_elastic(lambda_, mu)
    return eng


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind == "segments":
        mu, x, width, fric, y = _segments(case, seed)
        eng = Engine(0)
        eng.set_antiplane(mu, x, width, np.full(width.size, math.pi / 2))
        eng.set_friction(*fric)
        if width.size == 1:
            eng.set_kernel(_spring(mu, width))
        else:
            eng.buildG()
        s.update(eng=eng, y=y)
    elif kind in ("fault", "host_step"):
        m, friction, y = _fault(case, seed)
        eng = _engine(m.lambda_, m.mu)
        (eng.set_rectangles if case["mesh"] == "rectangles" else eng.set_triangles)(*m.geometry())
        eng.set_friction(*friction)
        eng.buildG(PRECISION[case.get("precision", "f64")])
        s.update(eng=eng, y=y)
    elif kind == "rectangles":
        s.update(model=_thrust(case["nx"], case["nz"], seed))
        s.update(eng=_engine(s["model"].lambda_, s["model"].mu))
    elif kind == "triangles":
        s.update(model=_mesh(case["nx"], case["ny"], seed))
        s.update(eng=_engine(s["model"].lambda_, s["model"].mu))
    elif kind == "volumes":
        fault, vol = _volume_model(case, seed)
        s.update(model=fault, vol=vol, eng=_engine(fault.lambda_, fault.mu))
    else:
        eng = Engine(0)
        ens = Ensemble(eng, PRECISION[case["precision"]])
        for g, (nx, nz) in enumerate(_groups(case)):
            m = _thrust(nx, nz, seed + 1000 * g)
            d, y = _instances(m, case["instances"], seed + 1000 * g)
            ens.add_group(m, d["a"], d["b"], d["sig"], d["L"], y)
        ens.build()
        s.update(eng=eng, ens=ens)
    return s


class _DeviceMatrix:
    """K where the engine keeps it (``Engine.kernel_dev_ptr``); a tensor on it
    keeps the engine."""

    def __init__(self, eng):
        self.eng = eng
        self.__cuda_array_interface__ = {"shape": eng.shape, "typestr": "<f8",
                                         "data": (eng.kernel_dev_ptr(), False), "version": 3}


def _parts(y, width):
    """A state vector (or several) as the parts that it consists of."""
    y = y.reshape(-1, y.shape[-1] // width, width) if y.ndim > 1 else y.reshape(-1, width)
    if width == 4:
        return {"slip": y[..., :1], "traction": y[..., 1:2], "theta": y[..., 2], "rate": y[..., 3]}
    return {"slip": y[..., :2], "traction": y[..., 2:5], "theta": y[..., 5], "rate": y[..., 6]}


def run(s):
    case, kind, eng = s["case"], s["kind"], s["eng"]
    if kind in ("segments", "fault"):
        r = eng.integrate(s["y"], NEVER, max_steps=case["steps"], max_step=case["max_step"],
                          log_cap=case["steps"])
        return dict(_parts(r.y, 4 if kind == "segments" else 7), time=r.t_log, dt=r.dt_log,
                    vmax=r.vmax_log)
    if kind == "host_step":
        y, n, t, h = s["y"].copy(), s["y"].size, 0.0, 1.0e-3
        dydt, times = np.empty(n), np.empty(case["steps"])
        for k in range(case["steps"]):
            eng.odefun(n, t, y, dydt)
            yscal = np.abs(y) + np.abs(h * dydt) + 1.0e-30
            t, _, h = eng.RKQSm(n, t, y, dydt, yscal, h, maximumTimeStep=case["max_step"])
            times[k] = t
        return dict(_parts(y, 7), time=times)
    if kind == "ensemble":
        ens = s["ens"]
        ens.reset()
        ens.run(NEVER, max_attempts=case["attempts"], max_step=SHORT_STEP)
        out = []
        for g in range(len(ens.groups)):
            y, t = ens.state(g)[:2]
            out.append(dict(_parts(y, 7), time=t))
        return out
    if kind == "triangles":
        eng.set_triangles(*s["model"].geometry())
    else:
        eng.set_rectangles(*s["model"].geometry())
    if kind == "volumes":
        eng.set_volumes(*s["vol"].geometry())
    eng.buildG(PRECISION[case.get("precision", "f64")])
    return torch.as_tensor(_DeviceMatrix(eng), device="cuda")


# ---- work and tolerance ---------------------------------------------------

def _rhs(attempts, m, n, columns, entry, state):
    """Bytes and flops of `attempts` Cash-Karp attempts on an m x n kernel."""
    k = float(m) * n * entry
    reads = 6 * attempts if k > ON_CHIP else 1
    return {"bytes": reads * k + 2.0 * 8 * state * columns,
            "flops": 6.0 * attempts * (2.0 * m * n + 60.0 * state) * columns}


def work(case):
    kind = case["kind"]
    if kind == "segments":
        n = case["segments"]
        return _rhs(case["steps"], n, n, 1, 8, 4 * n)
    if kind in ("fault", "host_step"):
        N = case["nx"] * case["nz"] * (2 if case["mesh"] == "triangles" else 1)
        entry = 8 if case.get("precision", "f64") == "f64" else 4
        return _rhs(case["steps"], 3 * N, 2 * N, 1, entry, 7 * N)
    if kind == "ensemble":
        total = {"bytes": 0.0, "flops": 0.0}
        entry = {"f64": 8, "bf16_i8": 3}.get(case["precision"], 4)
        for nx, nz in _groups(case):
            N = nx * nz
            w = _rhs(case["attempts"], 3 * N, 2 * N, case["instances"], entry, 7 * N)
            total = {k: total[k] + w[k] for k in total}
        return total
    # flops of one pair: the published closed forms evaluated once for both
    # unit slips (six unit strains) with their gradients
    if kind == "rectangles":
        N = case["nx"] * case["nz"]
        return {"bytes": 8.0 * 6 * N * N, "flops": 5000.0 * N * N}
    if kind == "triangles":
        N = 2 * case["nx"] * case["ny"]
        return {"bytes": 8.0 * 6 * N * N, "flops": 15000.0 * N * N}
    N, V = case["nx"] * case["nz"], case["vx"] * case["vy"] * case["vz"]
    return {"bytes": 8.0 * (3 * N + 6 * V) * (2 * N + 6 * V),
            "flops": 5000.0 * N * (N + V) + 50000.0 * V * (N + V)}


def tolerance(case):
    kind = case["kind"]
    if kind == "segments":
        return {"rel": 1e-9}
    if kind in ("fault", "host_step"):
        # through DC3D's binary32 results in K, or without them
        return {"rel": 4e-8 if case["mesh"] == "rectangles" else 1e-9}
    if kind == "ensemble":
        return {"rel": 1e-11 if case["precision"] == "f64" else 1e-9}
    if kind == "rectangles":
        # K is binary32 where it is formed, and largest next to the diagonal
        return {"rel": 2e-7, "max": 1e-4}
    return {"rel": 1e-13, "max": 1e-10} if kind == "triangles" else {"rel": 1e-11, "max": 1e-8}


# ---- the same in 64 bits --------------------------------------------------

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device=DEVICE)


def _dc3d_gradient(alpha, sd, cd, x, y, z, depth, al, aw):
    """Okada's DC3D: the nine displacement derivatives (uxx, uyx, uzx, uxy, ...)
    at (x, y, z) of unit strike and unit dip slip on [0, al] x [-aw, 0]."""
    a1, a2, a3, a4, a5 = (1 - alpha) / 2, alpha / 2, (1 - alpha) / alpha, 1 - alpha, alpha
    eps = 1e-6
    snap = lambda v: torch.where(v.abs() < eps, torch.zeros_like(v), v)  # noqa: E731
    total = [[0.0] * 9, [0.0] * 9]
    for image in (False, True):
        d0 = depth - z if image else depth + z
        p, q = y * cd + d0 * sd, snap(y * sd - d0 * cd)
        for k, et in enumerate((snap(p + aw), snap(p))):
            for j, xi in enumerate((snap(x), snap(x - al))):
                r2 = xi * xi + et * et + q * q
                r = r2.sqrt()
                r3, r5 = r * r2, r * r2 * r2
                yt, dt = et * cd + q * sd, et * sd - q * cd
                x11, y11 = 1 / (r * (r + xi)), 1 / (r * (r + et))
                x32, y32 = (2 * r + xi) * x11 * x11 / r, (2 * r + et) * y11 * y11 / r
                xx, xy, qx, qy = xi * xi, xi * y11, q * x11, q * y11
                ey, ez = sd / r - yt * q / r3, cd / r + dt * q / r3
                fy, fz = dt / r3 + xx * y32 * sd, yt / r3 + xx * y32 * cd
                gy, gz = 2 * x11 * sd - yt * q * x32, 2 * x11 * cd + dt * q * x32
                A = ([-a1 * qy - a2 * xx * q * y32, -a2 * xi * q / r3,
                      a1 * xy + a2 * xi * q * q * y32,
                      a1 * xy * sd + a2 * xi * fy + dt / 2 * x11, a2 * ey,
                      a1 * (cd / r + qy * sd) - a2 * q * fy,
                      a1 * xy * cd + a2 * xi * fz + yt / 2 * x11, a2 * ez,
                      -a1 * (sd / r - qy * cd) - a2 * q * fz],
                     [-a2 * xi * q / r3, -qy / 2 - a2 * et * q / r3, a1 / r + a2 * q * q / r3,
                      a2 * ey, a1 * dt * x11 + xy / 2 * sd + a2 * et * gy,
                      a1 * yt * x11 - a2 * q * gy,
                      a2 * ez, a1 * yt * x11 + xy / 2 * cd + a2 * et * gz,
                      -a1 * dt * x11 - a2 * q * gz])
                sign = 1.0 if j == k else -1.0
                if not image:
                    for s in range(2):
                        for i in (0, 3, 6):
                            u, v, w = A[s][i:i + 3]
                            f = sign if i == 6 else -sign
                            total[s][i] = total[s][i] + f * u
                            total[s][i + 1] = total[s][i + 1] + f * (v * cd - w * sd)
                            total[s][i + 2] = total[s][i + 2] + f * (v * sd + w * cd)
                    continue
                rd = r + dt
                d11 = 1 / (r * rd)
                j2, j5 = xi * yt / rd * d11, -(dt + yt * yt / rd) * d11
                k1, k3 = xi * (d11 - y11 * sd) / cd, (qy - yt * d11) / cd
                j3, j6 = (k1 - j2 * sd) / cd, (k3 - j5 * sd) / cd
                k2, k4 = 1 / r + k3 * sd, xy * cd - k1 * sd
                j1, j4 = j5 * cd - j6 * sd, -xy - j2 * cd + j3 * sd
                sc = a3 * sd * cd
                B = ([xx * q * y32 - a3 * j1 * sd, xi * q / r3 - a3 * j2 * sd,
                      -xi * q * q * y32 - a3 * j3 * sd,
                      -xi * fy - dt * x11 + a3 * (xy + j4) * sd, -ey + a3 * (1 / r + j5) * sd,
                      q * fy - a3 * (qy - j6) * sd,
                      -xi * fz - yt * x11 + a3 * k1 * sd, -ez + a3 * yt * d11 * sd,
                      q * fz + a3 * k2 * sd],
                     [xi * q / r3 + sc * j4, et * q / r3 + qy + sc * j5, -q * q / r3 + sc * j6,
                      -ey + sc * j1, -et * gy - xy * sd + sc * j2, q * gy + sc * j3,
                      -ez - sc * k3, -et * gz - xy * cd - sc * xi * d11, q * gz - sc * k4])
                c = dt + z
                x53 = (8 * r2 + 9 * r * xi + 3 * xx) * x11 ** 3 / r2
                y53 = (8 * r2 + 9 * r * et + 3 * et * et) * y11 ** 3 / r2
                h = q * cd - z
                z32, z53 = sd / r3 - h * y32, 3 * sd / r5 - h * y53
                y0, z0 = y11 - xx * y32, z32 - xx * z53
                py, pz = cd / r3 + q * y32 * sd, sd / r3 - q * y32 * cd
                qq = z * y32 + z32 + z0
                qqy = 3 * c * dt / r5 - qq * sd
                qqz = 3 * c * yt / r5 - qq * cd + q * y32
                qr, cdr, yy0 = 3 * q / r5, (c + dt) / r3, yt / r3 - y0 * cd
                c1 = a4 * (cd / r + 2 * qy * sd) - a5 * c * q / r3
                c2 = a4 * qy * cd - a5 * (c * et / r3 - z * y11 + xx * z32)
                e1 = a4 * yt * x11 - a5 * c * et * q * x32
                e2 = -dt * x11 - xy * sd - a5 * c * (x11 - q * q * x32)
                C = ([a4 * y0 * cd - a5 * q * z0,
                      -a4 * xi * (cd / r3 + 2 * q * y32 * sd) + a5 * c * xi * qr,
                      -a4 * xi * q * y32 * cd + a5 * xi * (3 * c * et / r5 - qq),
                      -a4 * xi * py * cd - a5 * xi * qqy,
                      a4 * 2 * (dt / r3 - y0 * sd) * sd - yt / r3 * cd
                      - a5 * (cdr * sd - et / r3 - c * yt * qr),
                      -a4 * q / r3 + yy0 * sd
                      + a5 * (cdr * cd + c * dt * qr - (y0 * cd + q * z0) * sd),
                      a4 * xi * pz * cd - a5 * xi * qqz,
                      a4 * 2 * (yt / r3 - y0 * cd) * sd + dt / r3 * cd
                      - a5 * (cdr * cd + c * dt * qr),
                      yy0 * cd - a5 * (cdr * sd - c * yt * qr - y0 * sd * sd + q * z0 * cd)],
                     [-a4 * xi / r3 * cd + a5 * c * xi * qr + xi * q * y32 * sd,
                      -a4 * yt / r3 + a5 * c * et * qr,
                      dt / r3 - y0 * sd + a5 * c / r3 * (1 - 3 * q * q / r2),
                      -a4 * et / r3 + y0 * sd * sd - a5 * (cdr * sd - c * yt * qr),
                      a4 * (x11 - yt * yt * x32)
                      - a5 * c * ((dt + 2 * q * cd) * x32 - yt * et * q * x53),
                      xi * py * sd + yt * dt * x32
                      + a5 * c * ((yt + 2 * q * sd) * x32 - yt * q * q * x53),
                      -q / r3 + y0 * sd * cd - a5 * (cdr * cd + c * dt * qr),
                      a4 * yt * dt * x32
                      - a5 * c * ((yt - 2 * q * sd) * x32 + dt * et * q * x53),
                      -xi * pz * sd + x11 - dt * dt * x32
                      - a5 * c * ((dt - 2 * q * cd) * x32 - dt * q * q * x53)])
                value = ([a4 * xy * cd - a5 * xi * q * z32, c1, c2],
                         [a4 * cd / r - qy * sd - a5 * c * q / r3, e1, e2])
                for s in range(2):
                    for i in (0, 3, 6):
                        a, b, cc = A[s][i:i + 3], B[s][i:i + 3], C[s][i:i + 3]
                        ab = [a[m] + b[m] for m in range(3)]
                        u = ab[0] + z * cc[0]
                        v = (ab[1] + z * cc[1]) * cd - (ab[2] + z * cc[2]) * sd
                        w = (ab[1] - z * cc[1]) * sd + (ab[2] - z * cc[2]) * cd
                        if i == 6:
                            f = value[s]
                            u, v = u + f[0], v + f[1] * cd - f[2] * sd
                            w = w - f[1] * sd - f[2] * cd
                        total[s][i] = total[s][i] + sign * u
                        total[s][i + 1] = total[s][i + 1] + sign * v
                        total[s][i + 2] = total[s][i + 2] + sign * w
    return [[v / (2 * math.pi) for v in t] for t in total]


def _f32(v):
    return v.to(torch.float32).to(torch.float64)


def _okada_kernel(m):
    """K (3N x 2N) of a fault of rectangles that strike north: tractions in the
    strike, dip and normal directions.  The coordinates and sizes go through
    binary32, as DC3D's arguments do; what it returns does not."""
    N = m.n
    dip = float(m.dip[0])
    one = torch.zeros((), dtype=torch.float64, device=DEVICE)
    degrees = float(np.float32(dip * 57.29577951308232))
    sd, cd = math.sin(degrees * (2 * math.pi / 360)), math.cos(degrees * (2 * math.pi / 360))
    alpha = float(np.float32((m.lambda_ + m.mu) / (m.lambda_ + 2 * m.mu)))
    x, L, W = _t(m.x), _t(m.length), _t(m.width)
    sv = torch.tensor([1.0, 0.0, 0.0], dtype=torch.float64, device=DEVICE)
    dv = torch.tensor([0.0, -math.cos(dip), -math.sin(dip)], dtype=torch.float64, device=DEVICE)
    nv = torch.tensor([0.0, math.sin(dip), -math.cos(dip)], dtype=torch.float64, device=DEVICE)
    xc = x + L[:, None] / 2 * sv - W[:, None] / 2 * dv
    K = torch.empty((3 * N, 2 * N), dtype=torch.float64, device=DEVICE)
    depth, al, aw = _f32(x[:, 2]), _f32(L), _f32(W)
    rows = max(1, min(N, (1 << 21) // N))
    for r0 in range(0, N, rows):
        c = xc[r0:r0 + rows]
        X = _f32(c[:, 0, None] - x[None, :, 0])
        Y = _f32(-(c[:, 1, None] - x[None, :, 1]))
        Z = _f32(-c[:, 2, None]) + one
        both = _dc3d_gradient(alpha, sd, cd, X, Y, Z, depth, al, aw)
        for s, g in enumerate(both):
            uxx, uyx, uzx, uxy, uyy, uzy, uxz, uyz, uzz = g
            # to north, east, down (strike north); e13 and e23 as okada92.f90
            # forms them
            e11, e22, e33 = uxx, uyy, uzz
            e12 = (-uxy - uyx) / 2
            e13, e23 = (-uxz - uzx) / 2, (uyz + uzy) / 2
            tr = m.lambda_ * (e11 + e22 + e33)
            S = {(0, 0): tr + 2 * m.mu * e11, (1, 1): tr + 2 * m.mu * e22,
                 (2, 2): tr + 2 * m.mu * e33, (0, 1): 2 * m.mu * e12, (0, 2): 2 * m.mu * e13,
                 (1, 2): 2 * m.mu * e23}
            full = lambda i, j: S[(min(i, j), max(i, j))]  # noqa: E731
            trac = [sum(full(i, j) * nv[j] for j in range(3)) for i in range(3)]
            for k, axis in enumerate((sv, dv, nv)):
                K[3 * r0 + k:3 * (r0 + c.shape[0]):3, s::2] = sum(trac[i] * axis[i]
                                                                 for i in range(3))
    return K


def _angular(x, y, z, alpha, b, nu):
    """Angular dislocation without the Burgers function (Nikkhoo and Walter
    2015): displacement for the Burgers vector b, in its own frame."""
    ca, sa = torch.cos(alpha), torch.sin(alpha)
    eta, zeta = y * ca - z * sa, y * sa + z * ca
    r = (x * x + y * y + z * z).sqrt()
    zeta, z = torch.minimum(zeta, r), torch.minimum(z, r)
    rz, rt = r - z, r - zeta
    lz, lt = rz.log(), rt.log()
    n = 1 - 2 * nu
    k = 1 / (8 * math.pi * (1 - nu))
    w = n * (ca * lt - lz)
    u = b[0] * (x * y / (r * rz) - x * eta / (r * rt)) \
        + b[1] * (x * x * ca / (r * rt) - x * x / (r * rz) - w) \
        + b[2] * sa * (n * lt - x * x / (r * rt))
    v = b[0] * (eta * sa / rt - y * eta / (r * rt) + y * y / (r * rz) + w) \
        + b[1] * x * (y * ca / (r * rt) - sa * ca / rt - y / (r * rz)) \
        + b[2] * sa * x * (sa / rt - y / (r * rt))
    t = b[0] * (eta * ca / rt - y / r - eta * z / (r * rt) - n * sa * lt) \
        + b[1] * x * (z * ca / (r * rt) - ca * ca / rt + 1 / r) \
        + b[2] * sa * x * (ca / rt - z / (r * rt))
    return k * u, k * v, k * t


def _harmonic(y1, y2, y3, beta, b, nu, a):
    """Harmonic correction of an angular dislocation at depth a (Nikkhoo and
    Walter 2015, appendix): displacement for the Burgers vector b."""
    sb, cb = torch.sin(beta), torch.cos(beta)
    cot, half = cb / sb, torch.cos(beta / 2) / torch.sin(beta / 2)
    y3b = y3 + 2 * a
    z1, z3 = y1 * cb + y3b * sb, -y1 * sb + y3b * cb
    r = (y1 * y1 + y2 * y2 + y3b * y3b).sqrt()
    r2, r3 = r * r, r * r * r
    f = 2 * torch.atan(-y2 / (-(r + y3b) * half + y1))
    n, m = 1 - 2 * nu, 1 - nu
    p, q, d = r + y3b, r + z3, y3b - a            # p: W6, q: W7
    lp, lq = p.log(), q.log()
    g, s, c2 = r * cb + y3b, r * sb - y1, cot * cot
    v11 = -2 * m * n * f * c2 + n * y2 / p * ((n - a / r) * cot - y1 / p * (nu + a / r)) \
        + n * y2 * cb * cot / q * (cb + a / r) + a * y2 * d * cot / r3 \
        + y2 * d / (r * p) * (-n * cot + y1 / p * (2 * nu + a / r) + a * y1 / r2) \
        + y2 * d / (r * q) * (cb / q * (g * (n * cb - a / r) * cot + 2 * m * s * cb)
                              - a * y3b * cb * cot / r2)
    v21 = n * ((2 * m * c2 - nu) * lp - (2 * m * c2 + n) * cb * lq) \
        - n / p * (y1 * cot * (n - a / r) + nu * y3b - a + y2 * y2 / p * (nu + a / r)) \
        - n * z1 * cot / q * (cb + a / r) - a * y1 * d * cot / r3 \
        + d / p * (-2 * nu + (n * y1 * cot - a) / r + y2 * y2 / (r * p) * (2 * nu + a / r)
                   + a * y2 * y2 / r3) \
        + d / q * (cb * cb - (n * z1 * cot + a * cb) / r + a * y3b * z1 * cot / r3
                   - (y2 * y2 * cb * cb - a * z1 * cot / r * g) / (r * q))
    v31 = 2 * m * (n * f * cot + y2 / p * (2 * nu + a / r) - y2 * cb / q * (cb + a / r)) \
        + y2 * d / r * (2 * nu / p + a / r2) \
        + y2 * d * cb / (r * q) * (n - g / q * (cb + a / r) - a * y3b / r2)
    v12 = n * ((2 * m * c2 + nu) * lp - (2 * m * c2 + 1) * cb * lq) \
        + n / p * (-n * y1 * cot + nu * y3b - a + a * y1 * cot / r + y1 * y1 / p * (nu + a / r)) \
        - n * cot / q * (z1 * cb - a * s / (r * cb)) - a * y1 * d * cot / r3 \
        + d / p * (2 * nu + (n * y1 * cot + a) / r - y1 * y1 / (r * p) * (2 * nu + a / r)
                   - a * y1 * y1 / r3) \
        + d * cot / q * (-cb * sb + a * y1 * y3b / (r3 * cb)
                         + s / r * (2 * m * cb - g / q * (1 + a / (r * cb))))
    v22 = 2 * m * n * f * c2 + n * y2 / p * (-(n - a / r) * cot + y1 / p * (nu + a / r)) \
        - n * y2 * cot / q * (1 + a / (r * cb)) - a * y2 * d * cot / r3 \
        + y2 * d / (r * p) * (n * cot - 2 * nu * y1 / p - a * y1 / r * (1 / r + 1 / p)) \
        + y2 * d * cot / (r * q) * (-2 * m * cb + g / q * (1 + a / (r * cb))
                                    + a * y3b / (r2 * cb))
    v32 = -2 * m * n * cot * (lp - cb * lq) - 2 * m * y1 / p * (2 * nu + a / r) \
        + 2 * m * z1 / q * (cb + a / r) + d / r * (n * cot - 2 * nu * y1 / p - a * y1 / r2) \
        - d / q * (cb * sb + g * cot / r * (2 * m * cb - g / q)
                   + a / r * (sb - y3b * z1 / r2 - z1 * g / (r * q)))
    v13 = n * (y2 / p * (1 + a / r) - y2 * cb / q * (cb + a / r)) - y2 * d / r * (a / r2 + 1 / p) \
        + y2 * d * cb / (r * q) * (g / q * (cb + a / r) + a * y3b / r2)
    v23 = n * (-sb * lq - y1 / p * (1 + a / r) + z1 / q * (cb + a / r)) \
        + y1 * d / r * (a / r2 + 1 / p) \
        - d / q * (sb * (cb - a / r) + z1 / r * (1 + a * y3b / r2)
                   - (y2 * y2 * cb * sb - a * z1 / r * g) / (r * q))
    v33 = 2 * m * f + 2 * m * y2 * sb / q * (cb + a / r) \
        + y2 * d * sb / (r * q) * (1 + g / q * (cb + a / r) + a * y3b / r2)
    k = 1 / (4 * math.pi * m)
    return (k * (b[0] * v11 + b[1] * v12 + b[2] * v13), k * (b[0] * v21 + b[1] * v22 + b[2] * v23),
            k * (b[0] * v31 + b[1] * v32 + b[2] * v33))


def _dot(a, b):
    return sum(a[i] * b[i] for i in range(3))


def _cross(a, b):
    return [a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]


def _unit(a):
    n = _dot(a, a).sqrt()
    return [v / n for v in a]


def _tri_frame(P):
    """Normal, strike and dip directions (east, north, up)."""
    n = _unit(_cross([P[1][i] - P[0][i] for i in range(3)], [P[2][i] - P[0][i] for i in range(3)]))
    zero = torch.zeros_like(n[0])
    s = _unit([-n[1], n[0], zero])
    return n, s, _cross(n, s)


def _tri_full(X, P, slip, nu):
    """Displacement of a triangle in the full space; slip (normal, strike, dip)."""
    axes = _tri_frame(P)
    local = lambda v: [_dot(a, [v[i] - P[1][i] for i in range(3)]) for a in axes]  # noqa: E731
    x, y, z = local(X)
    _, y1, z1 = local(P[0])
    _, y3, z3 = local(P[2])
    zero = torch.zeros_like(y1)
    V = [(y1, z1), (zero, zero), (y3, z3)]
    e = lambda a, b: [(V[b][i] - V[a][i]) / ((V[b][0] - V[a][0]) ** 2  # noqa: E731
                                             + (V[b][1] - V[a][1]) ** 2).sqrt() for i in range(2)]
    e12, e13, e23 = e(0, 1), e(0, 2), e(1, 2)
    dot = lambda a, b: a[0] * b[0] + a[1] * b[1]  # noqa: E731
    angles = [torch.acos(dot(e12, e13)), torch.acos(-dot(e12, e23)), torch.acos(dot(e23, e13))]
    # the configuration (sign of the side vectors) from barycentric coordinates
    den = (0 - z3) * (y1 - y3) + y3 * (z1 - z3)
    A = ((0 - z3) * (y - y3) + y3 * (z - z3)) / den
    B = ((z3 - z1) * (y - y3) + (y1 - y3) * (z - z3)) / den
    C = 1 - A - B
    flip = ((A <= 0) & (B > C) & (C > A)) | ((B <= 0) & (C > A) & (A > B)) \
        | ((C <= 0) & (A > B) & (B > C))
    sign = torch.where(flip, -1.0, 1.0).detach()
    u = [torch.zeros_like(x) for _ in range(3)]
    for v, (side, f) in enumerate(((e13, -1.0), (e12, 1.0), (e23, 1.0))):
        s1, s2 = sign * f * side[0], sign * f * side[1]
        ty, tz = y - V[v][0], z - V[v][1]
        b = (slip[0], s2 * slip[1] - s1 * slip[2], s1 * slip[1] + s2 * slip[2])
        d = _angular(x, s2 * ty - s1 * tz, s1 * ty + s2 * tz, -math.pi + angles[v], b, nu)
        u[0] = u[0] + d[0]
        u[1] = u[1] + s2 * d[1] + s1 * d[2]
        u[2] = u[2] - s1 * d[1] + s2 * d[2]
    a, b, c = [-x, y1 - y, z1 - z], [-x, -y, -z], [-x, y3 - y, z3 - z]
    na, nb, nc = (_dot(v, v).sqrt() for v in (a, b, c))
    solid = torch.atan2(_dot(a, _cross(b, c)), na * nb * nc + _dot(a, b) * nc + _dot(a, c) * nb
                        + _dot(b, c) * na)
    u = [u[i] - slip[i] * solid / (2 * math.pi) for i in range(3)]
    return [sum(axes[k][i] * u[k] for k in range(3)) for i in range(3)]


def _tri_harmonic(X, P, slip, nu):
    axes = _tri_frame(P)
    bX = [sum(axes[k][i] * slip[k] for k in range(3)) for i in range(3)]
    u = [torch.zeros_like(X[0]) for _ in range(3)]
    for A, B in ((0, 1), (1, 2), (2, 0)):
        side = [P[B][i] - P[A][i] for i in range(3)]
        beta = torch.acos(-side[2] / _dot(side, side).sqrt())
        zero = torch.zeros_like(beta)
        h = _unit([side[0], side[1], zero])
        frame = (h, [h[1], -h[0], zero], [zero, zero, zero - 1])
        yA = [_dot(a, [X[i] - P[A][i] for i in range(3)]) for a in frame]
        sA = [_dot(a, side) for a in frame]
        bA = [_dot(a, bX) for a in frame]
        angle = torch.where(beta * yA[0] >= 0, -math.pi + beta, beta).detach()
        wA = _harmonic(*yA, angle, bA, nu, -P[A][2])
        wB = _harmonic(*[yA[i] - sA[i] for i in range(3)], angle, bA, nu, -P[B][2])
        for i in range(3):
            u[i] = u[i] + sum(frame[k][i] * (wB[k] - wA[k]) for k in range(3))
    return u


def _triangle_kernel(m):
    """K (3N x 2N) of a mesh of triangles: strain by forward-mode
    differentiation of the displacement."""
    nu = m.lambda_ / (m.lambda_ + m.mu) / 2
    v = _t(m.vertices)
    idx = [torch.as_tensor(np.asarray(i, dtype=np.int64) - 1, device=DEVICE)
           for i in (m.i1, m.i2, m.i3)]
    ned = [[v[i][:, k] for k in range(3)] for i in idx]
    xc = [(ned[0][k] + ned[1][k] + ned[2][k]) / 3 for k in range(3)]
    n = _unit(_cross([ned[1][k] - ned[0][k] for k in range(3)],
                     [ned[2][k] - ned[0][k] for k in range(3)]))
    n = [torch.where(n[2] > 0, -c, c) for c in n]       # upwards
    h = (n[0] ** 2 + n[1] ** 2).sqrt()
    s = [n[1] / h, -n[0] / h, torch.zeros_like(h)]
    d = [n[1] * s[2] - n[2] * s[1], n[2] * s[0] - n[0] * s[2], n[0] * s[1] - n[1] * s[0]]
    P = [[q[1], q[0], -q[2]] for q in ned]              # east, north, up
    M = [[q[0], q[1], -q[2]] for q in P]
    N = m.n
    K = torch.empty((3 * N, 2 * N), dtype=torch.float64, device=DEVICE)
    rows = max(1, min(N, (1 << 22) // N))
    for r0 in range(0, N, rows):
        r = slice(r0, min(N, r0 + rows))
        X = [xc[1][r, None].expand(-1, N), xc[0][r, None].expand(-1, N),
             -xc[2][r, None].expand(-1, N)]
        X = [a.contiguous() for a in X]
        for c, slip in enumerate(((0.0, 1.0, 0.0), (0.0, 0.0, -1.0))):
            def u(*x):
                f, g = _tri_full(x, P, slip, nu), _tri_full(x, M, slip, nu)
                w = _tri_harmonic(x, P, slip, nu)
                return tuple(f[i] + g[i] + w[i] for i in range(3))
            grad = []
            for k in range(3):
                t = tuple(torch.ones_like(a) if i == k else torch.zeros_like(a)
                          for i, a in enumerate(X))
                grad.append(torch.func.jvp(u, tuple(X), t)[1])
            e = lambda i, j: (grad[i][j] + grad[j][i]) / 2  # noqa: E731
            tr = m.lambda_ * (grad[0][0] + grad[1][1] + grad[2][2])
            S = lambda i, j: 2 * m.mu * e(i, j) + (tr if i == j else 0.0)  # noqa: E731
            # receivers' axes in east, north, up
            ax = [[a[1][r, None], a[0][r, None], -a[2][r, None]] for a in (s, d, n)]
            trac = [sum(S(i, j) * ax[2][j] for j in range(3)) for i in range(3)]
            for k in range(3):
                K[3 * r0 + k:3 * r.stop:3, c::2] = sum(trac[i] * ax[k][i] for i in range(3))
    return K


def _antiplane_kernel(mu, x, width):
    """K of vertical segments in antiplane strain: a screw dislocation at each
    end and its image."""
    q, w = _t(x[:, 2]), _t(width)
    z = (q + w / 2)[:, None]
    return mu / (2 * math.pi) * (-1 / (z - q) + 1 / (z + q) + 1 / (z - q - w) - 1 / (z + q + w))


_CK = ((0.2,), (3 / 40, 9 / 40), (0.3, -0.9, 1.2), (-11 / 54, 2.5, -70 / 27, 35 / 27),
       (1631 / 55296, 175 / 512, 575 / 13824, 44275 / 110592, 253 / 4096))
_C5 = (37 / 378, 0.0, 250 / 621, 125 / 594, 0.0, 512 / 1771)
_DC = (37 / 378 - 2825 / 27648, 0.0, 250 / 621 - 18575 / 48384, 125 / 594 - 13525 / 55296,
       -277 / 14336, 512 / 1771 - 0.25)


def _rhs_fault(K, f):
    """odefun of B instances of a 3-D fault; states are (B, N, 7)."""
    ln = math.log(10.0)

    def rhs(y):
        rake = torch.atan2(y[..., 3], y[..., 2])
        V = torch.exp(y[..., 6] * ln)
        cr, sr = torch.cos(rake), torch.sin(rake)
        v = torch.stack([V * cr - f["vplc"], V * sr - f["vpls"]], -1)
        t = (v.reshape(v.shape[0], -1) @ K.T).reshape(*V.shape, 3)
        out = torch.empty_like(y)
        out[..., 0], out[..., 1] = V * cr, V * sr
        out[..., 5] = (torch.exp(-y[..., 5] * ln) - V / f["L"]) / ln
        dtau = t[..., 0] * cr + t[..., 1] * sr
        out[..., 6] = (dtau - f["b"] * f["sig"] * out[..., 5] * ln) \
            / (f["a"] * f["sig"] + f["damping"] * V) / ln
        corr = f["damping"] * V * out[..., 6] * ln
        out[..., 2], out[..., 3], out[..., 4] = t[..., 0] - corr * cr, t[..., 1] - corr * sr, \
            t[..., 2]
        return out, V
    return rhs


def _rhs_segments(K, f):
    ln = math.log(10.0)

    def rhs(y):
        V = torch.exp(y[..., 3] * ln)
        t = (V - f["vplc"]) @ K.T
        out = torch.empty_like(y)
        out[..., 0] = V
        out[..., 2] = (torch.exp(-y[..., 2] * ln) - V / f["L"]) / ln
        out[..., 3] = (t - f["b"] * f["sig"] * out[..., 2] * ln) \
            / (f["a"] * f["sig"] + f["damping"] * V) / ln
        out[..., 1] = t - f["damping"] * V * out[..., 3] * ln
        return out, V
    return rhs


def _rk45(rhs, y, max_step, steps=None, attempts=None, epsilon=1e-6):
    """RKQS over Cash-Karp steps for B instances in lockstep: each until its
    number of accepted steps, or of attempts.  Returns the states, the times
    and the logs (time, step, vMax at the step's start) of instance 0."""
    B = y.shape[0]
    one = torch.ones(B, dtype=torch.float64, device=y.device)
    h, time, done = 1e-3 * one, 0.0 * one, torch.zeros(B, dtype=torch.int64, device=y.device)
    k1 = scale = None
    new = torch.ones(B, dtype=torch.bool, device=y.device)
    vmax, log, tried = 0.0 * one, [], 0
    c = lambda v: v[:, None, None]  # noqa: E731
    while (int(done.min()) < steps) if attempts is None else (tried < attempts):
        tried += 1
        d, V = rhs(y)
        s = y.abs() + (c(h) * d).abs() + 1e-30
        if k1 is None:
            k1, scale, vmax = d, s, V.amax(1)
        else:
            k1, scale = torch.where(c(new), d, k1), torch.where(c(new), s, scale)
            vmax = torch.where(new, V.amax(1), vmax)
        ks = [k1]
        for row in _CK:
            ks.append(rhs(y + c(h) * sum(b * k for b, k in zip(row, ks)))[0])
        cand = y + c(h) * sum(b * k for b, k in zip(_C5, ks))
        err = (c(h) * sum(b * k for b, k in zip(_DC, ks)) / scale).abs().amax((1, 2)) / epsilon
        new = err <= 1.0
        y = torch.where(c(new), cand, y)
        time = torch.where(new, time + h, time)
        if bool(new[0]):
            log.append((float(time[0]), float(h[0]), float(vmax[0])))
        grow = torch.where(err > 1.89e-4, 0.7 * h * err.clamp(min=1e-300) ** -0.2, 10.0 * h)
        h = torch.where(new, grow.clamp(max=max_step), 0.7 * h * err.clamp(min=1e-300) ** -0.15)
        done = done + new
    return y, time, np.array(log)


def _friction(sig, a, b, L, damping, vplc, vpls=None):
    f = {"sig": sig, "a": a, "b": b, "L": L, "damping": damping, "vplc": vplc}
    f = {k: _t(v) for k, v in f.items()}
    if vpls is not None:
        f["vpls"] = _t(vpls)
    return f


def _exact_instances(m, count, seed):
    d, y = _instances(m, count, seed)
    f = _friction(d["sig"], d["a"], d["b"], d["L"], m.damping, m.Vpl * np.cos(m.rake),
                  m.Vpl * np.sin(m.rake))
    return f, _t(y.reshape(count, m.n, 7))


def exact(case, seed):
    kind = case["kind"]
    if kind == "segments":
        mu, x, width, fric, y = _segments(case, seed)
        n = width.size
        K = _t(_spring(mu, width)) if n == 1 else _antiplane_kernel(mu, x, width)
        f = _friction(fric[3], fric[4], fric[5], fric[6], fric[8], fric[0])
        y, _, log = _rk45(_rhs_segments(K, f), _t(y.reshape(1, n, 4)), case["max_step"],
                          steps=case["steps"])
        return dict(_parts(y[0].reshape(-1), 4), time=log[:, 0], dt=log[:, 1], vmax=log[:, 2])
    if kind in ("fault", "host_step"):
        m, fric, y = _fault(case, seed)
        f = _friction(fric[3], fric[4], fric[5], fric[6], fric[8], fric[0] * np.cos(fric[1]),
                      fric[0] * np.sin(fric[1]))
        K = (_okada_kernel if case["mesh"] == "rectangles" else _triangle_kernel)(m)
        y, _, log = _rk45(_rhs_fault(K, f), _t(y.reshape(1, m.n, 7)), case["max_step"],
                          steps=case["steps"])
        out = dict(_parts(y[0].reshape(-1), 7), time=log[:, 0])
        return out if kind == "host_step" else dict(out, dt=log[:, 1], vmax=log[:, 2])
    if kind == "ensemble":
        out = []
        for g, (nx, nz) in enumerate(_groups(case)):
            m = _thrust(nx, nz, seed + 1000 * g)
            f, y = _exact_instances(m, case["instances"], seed + 1000 * g)
            y, time, _ = _rk45(_rhs_fault(_okada_kernel(m), f), y, SHORT_STEP,
                               attempts=case["attempts"])
            y = y.reshape(y.shape[0], -1)
            for k in range(0, case["instances"], 64):       # the groups of 64 of one geometry
                out.append(dict(_parts(y[k:k + 64], 7), time=time[k:k + 64]))
        return out
    if kind == "rectangles":
        return _okada_kernel(_thrust(case["nx"], case["nz"], seed))
    if kind == "triangles":
        return _triangle_kernel(_mesh(case["nx"], case["ny"], seed))
    # without the closed forms of the strain volumes themselves, quadrature of
    # the half-space point sources over every volume: minutes
    return None
