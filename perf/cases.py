"""The estimator's timed cases.

Each case is one piece of work that a program built on this package hands to the GPU, called
through the public entry points: windows of single estimators (linear, time-varying and
extended), batches of independent estimators, a sliding-window bank, log-likelihood gradients,
marginal densities and relative-system prediction.  Systems, window lengths and grids are those
of the package's seeded workloads, of its tests and of its benchmark.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what the program holds before the call
    run(state)           one pass
    exact(case, seed)    the outputs that have a closed form, in 64 bits, by numpy alone
    work(case)           bytes and operations that one pass cannot do without
"""
import ctypes as ct

import numpy as np
import torch

from cauchyfriendly_amd import pycauchy
from cauchyfriendly_amd import workloads as W
from cauchyfriendly_amd.cauchy_estimator import (C_CauchyDynamicsUpdateContainer, Py_CauchyDynamicsUpdateContainer,
                                                 PyCauchyEstimator, eval_2d_relative_system_cpdf, step_estimators)
from cauchyfriendly_amd.likelihood import (scale_directions, tangent_gradients, theta_of, window_loglikelihood)

# Terms after a scalar update grow by about this factor from one update to the next, by state
# dimension and noise columns (the seeded systems and the reference's demos agree on them).
GROWTH = {(1, 1): 1.2, (2, 1): 2.7, (2, 2): 3.8, (3, 1): 3.4, (3, 2): 5.2, (4, 1): 3.9, (4, 2): 4.9, (5, 1): 4.1,
          (5, 2): 4.1, (6, 1): 4.2, (7, 1): 4.0, (8, 1): 6.0}
ORBIT_GROWTH = 5.6


# ------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # A tracker's ordinary window: one small LTI estimator over 8 steps.  Every update is a
        # few thousand terms at most, so launches and round trips decide.
        {"name": "window_lti3", "kind": "window", "mode": "lti", "states": 3, "noises": 1, "rows": 1, "steps": 8},
        # A larger state over a shorter window: many hyperplanes per term, few terms.
        {"name": "window_lti6", "kind": "window", "mode": "lti", "states": 6, "noises": 1, "rows": 1, "steps": 6},
        # The largest single estimator: 5-state LTV, two noises, two measurements per step,
        # 2.8 million terms at its last update.
        {"name": "window_ltv5", "kind": "window", "mode": "ltv", "states": 5, "noises": 2, "rows": 2, "steps": 5},
        # The longest window the engine takes at two states and two noises: 20 hyperplanes per
        # term, large cell tables.
        {"name": "window_ltv2", "kind": "window", "mode": "ltv", "states": 2, "noises": 2, "rows": 1, "steps": 10},
        # The extended (nonlinear) estimator on the pendulum, two measurements per step.
        {"name": "window_pendulum", "kind": "window", "mode": "nonlin", "states": 2, "noises": 1, "rows": 2,
         "steps": 6},
        # A few dozen independent targets stepped together.
        {"name": "batch_48", "kind": "batch", "estimators": 48, "groups": 2},
        # The ragged batch of the benchmark: states 2 to 5, windows of 4 to 8 steps, 30% of the
        # measurements impulsive.
        {"name": "batch_512", "kind": "batch", "estimators": 512, "groups": 4},
        # Maximum-likelihood tuning: the log-likelihood of many short records, forward and
        # backward, in all 14 parameters of a 3-state system.
        {"name": "gradient_64", "kind": "gradient", "sequences": 64, "steps": 6},
        # The 7-state orbit windows with their gradients in the noise scales.
        {"name": "orbit_8", "kind": "orbit", "windows": 8, "steps": 4},
        # A sliding-window bank from its first measurement through steady state.
        {"name": "bank_ltv5", "kind": "bank", "mode": "ltv", "states": 5, "noises": 2, "rows": 2, "windows": 5,
         "measurements": 9},
        # Plots and risk limits: the joint marginal density of two states on a grid, from an
        # estimator of about half a million terms.
        {"name": "marginal2d_101", "kind": "marginal2d", "states": 5, "noises": 2, "rows": 2, "steps": 5,
         "points": 101},
        # Conjunction screening: the relative position density of two estimators.
        {"name": "relative_21", "kind": "relative", "states": 5, "noises": 2, "rows": 2, "steps": 3, "points": 21},
    ]


# Window lengths that a drawn single estimator may have (steps low, steps high), by mode, state
# dimension, noises and measurement rows; none costs more than the listed windows.
WINDOWS = [("lti", 1, 1, 1, 4, 16), ("lti", 2, 1, 1, 5, 10), ("lti", 3, 1, 1, 4, 10), ("lti", 4, 1, 1, 3, 8),
           ("lti", 5, 1, 1, 3, 8), ("lti", 6, 1, 1, 3, 7), ("lti", 8, 1, 1, 2, 5), ("ltv", 2, 2, 1, 4, 9),
           ("ltv", 3, 2, 1, 3, 8), ("ltv", 4, 2, 2, 2, 4), ("ltv", 5, 2, 2, 2, 4), ("ltv", 7, 1, 2, 2, 4),
           ("nonlin", 2, 1, 1, 4, 9), ("nonlin", 2, 1, 2, 2, 6)]


def _log_int(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["window", "window", "window", "batch", "gradient", "orbit", "bank", "marginal1d", "marginal2d",
                       "relative"])
    if kind == "window":
        mode, n, noises, rows, low, high = rng.choice(WINDOWS)
        return {"kind": kind, "mode": mode, "states": n, "noises": noises, "rows": rows,
                "steps": rng.randint(low, high)}
    if kind == "batch":
        return {"kind": kind, "estimators": _log_int(rng, 3, 400), "groups": rng.randint(1, 4)}
    if kind == "gradient":
        return {"kind": kind, "sequences": _log_int(rng, 1, 60), "steps": rng.randint(3, 6)}
    if kind == "orbit":
        return {"kind": kind, "windows": rng.randint(1, 7), "steps": rng.randint(2, 4)}
    if kind == "bank":
        mode, n, noises, rows, wins = rng.choice([("lti", 3, 1, 1, 6), ("lti", 4, 1, 1, 5), ("ltv", 4, 2, 2, 3),
                                                  ("ltv", 5, 2, 2, 4)])
        windows = rng.randint(3, wins)
        return {"kind": kind, "mode": mode, "states": n, "noises": noises, "rows": rows, "windows": windows,
                "measurements": windows + rng.randint(1, 4)}
    n, noises, rows, low, high = rng.choice([(2, 1, 1, 3, 7), (3, 1, 1, 3, 7), (4, 1, 1, 3, 6), (5, 2, 2, 2, 4)])
    if kind == "relative":
        # pairs of terms: one step fewer than a density's estimator
        return {"kind": kind, "states": n, "noises": noises, "rows": rows, "steps": max(2, min(high - 2, low + 1)),
                "points": rng.randint(4, 25)}
    points = _log_int(rng, 31, 20001) if kind == "marginal1d" else _log_int(rng, 7, 101)
    return {"kind": kind, "states": n, "noises": noises, "rows": rows, "steps": rng.randint(low, high),
            "points": points}


# ------------------------------------------------------------------------------------ inputs
def _system(c, seed, steps):
    """The case's linear system: the 3-state recipe at any dimension, or the 5-state LTV one."""
    if c["mode"] == "lti":
        return W.lti_system(d=c["states"], steps=steps, seed_offset=seed)
    return W.ltv_system(d=c["states"], steps=steps, seed_offset=seed, pncc=c["noises"], p=c["rows"])


def _with_mode(c):
    return dict(c, mode="ltv" if c["noises"] > 1 or c["rows"] > 1 else "lti")


def _dynamics(s):
    """The LTV callback: writes Phi of the step ahead."""
    def update(c_duc):
        duc = Py_CauchyDynamicsUpdateContainer(c_duc)
        k = max(duc.cget_step(), 0)
        duc.cset_Phi(s.Phi(k))
        c_duc.contents.step = k + 1
    return update


def _srand(seed):
    """The engine draws its root point and perturbation from glibc's rand() at creation."""
    ct.CDLL("libc.so.6").srand(ct.c_uint(seed))


def _estimator(s, window):
    _srand(s.srand_seed)
    if len(s.Phis) > 1:
        est = PyCauchyEstimator("ltv", window)
        est.initialize_ltv(s.A0, s.p0, s.b0, s.Phi(0), None, s.Gamma, s.beta, s.H, s.gamma, _dynamics(s))
    else:
        est = PyCauchyEstimator("lti", window)
        est.initialize_lti(s.A0, s.p0, s.b0, s.Phi(0), None, s.Gamma, s.beta, s.H, s.gamma)
    return est


def _extended(pend, window):
    _srand(pend.srand_seed)
    est = PyCauchyEstimator("nonlin", window)
    est.initialize_nonlin(pend.xbar0, pend.A0, pend.p0, pend.b0, pend.beta, pend.gamma,
                          *pend.callbacks(Py_CauchyDynamicsUpdateContainer), 0, pend.dt)
    return est


def _batch_systems(count, seed):
    """Independent estimators of 2 to 5 states over windows of 4 to 8 steps, each combination in
    turn, with the benchmark's outliers."""
    return [W.lti_system(d=2 + j % 4, steps=4 + j // 4 % 5, seed_offset=seed + 1000 * (j + 1), outlier_prob=0.3,
                         outlier_scale=50.0) for j in range(count)]


def _stepped(s, steps):
    est = _estimator(s, steps + 1)
    for k in range(steps):
        est.step(s.zs[k])
    return est


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind, "case": case}
    if kind == "window":
        if case["mode"] == "nonlin":
            s = W.pendulum_system(p=case["rows"], steps=case["steps"], seed_offset=seed)
            state["start"] = (s.A0, s.p0, s.b0, s.xbar0)
            state["est"] = _extended(s, case["steps"])
        else:
            s = _system(case, seed, case["steps"])
            state["start"] = (s.A0, s.p0, s.b0)
            state["est"] = _estimator(s, case["steps"])
        state["zs"] = s.zs
        state["dynamics_step"] = _rewind(state["est"], case["mode"])
    elif kind == "batch":
        state["systems"] = _batch_systems(case["estimators"], seed)
        state["ests"] = [_estimator(s, s.num_steps) for s in state["systems"]]
    elif kind == "gradient":
        base = W.lti_sequences(case["sequences"], case["steps"], seed_offset=seed)
        state["systems"] = base
        state["theta"] = torch.tensor(np.array([theta_of(s) for s in base]), requires_grad=True)
        state["weight"] = torch.tensor(np.random.default_rng(seed).uniform(0.5, 1.5, case["sequences"]))
    elif kind == "orbit":
        state["systems"] = W.leo7_windows(case["windows"], case["steps"], dt=1.0, seed_offset=seed)
    elif kind == "bank":
        s = _system(case, seed, case["measurements"])
        state["system"] = s
        state["callback"] = ct.CFUNCTYPE(None, ct.POINTER(C_CauchyDynamicsUpdateContainer))(_dynamics(s))
    elif kind in ("marginal1d", "marginal2d"):
        state["est"] = _stepped(_system(_with_mode(case), seed, case["steps"] + 1), case["steps"])
        state["centre"], _ = state["est"].get_last_mean_cov()
    elif kind == "relative":
        c = _with_mode(case)
        state["primary"] = _stepped(_system(c, seed, case["steps"] + 1), case["steps"])
        state["secondary"] = _stepped(_system(c, seed + 500, case["steps"] + 1), case["steps"])
        T = np.zeros((2, case["states"]))
        T[0, 0] = T[1, case["states"] - 1] = 1.0
        state["T"] = T
    else:
        raise ValueError(f"unknown kind {kind}")
    return state


def _rewind(est, mode):
    """Puts the dynamics container's step counter of a time-varying window back to its start."""
    if mode == "lti":
        return lambda: None
    duc = ct.cast(pycauchy.pycauchy_single_step_get_duc(est.py_handle), ct.POINTER(C_CauchyDynamicsUpdateContainer))
    first = int(duc.contents.step)

    def rewind():
        duc.contents.step = first
    return rewind


# ------------------------------------------------------------------------------------ one pass
def _run_window(st):
    est = st["est"]
    est.reset(*st["start"])
    st["dynamics_step"]()
    rows = [est.step(z, full_info=True) for z in st["zs"]]
    n = len(rows)
    xs = [x for r in rows for x in r[0]]
    Ps = [P for r in rows for P in r[1]]
    info = est.moment_info
    return {"first": {"x": xs[0], "P": Ps[0]},
            "later": {"x": np.array(xs[1:]), "P": np.array(Ps[1:]), "fz": np.array(info["fz"][-n:]),
                      "err": np.array(info["err_code"][-n:])}}


def _run_batch(st):
    ests, systems = st["ests"], st["systems"]
    for e, s in zip(ests, systems):
        e.reset(s.A0, s.p0, s.b0)
    for k in range(max(s.num_steps for s in systems)):
        live = [i for i, s in enumerate(systems) if k < s.num_steps]
        step_estimators([ests[i] for i in live], [systems[i].zs[k] for i in live],
                        merged_groups=st["case"]["groups"])

    def gather(key, which):
        return np.concatenate([np.reshape(v, -1) for e, s in zip(ests, systems)
                               for v in e.moment_info[key][-s.num_steps:][which]])
    first, later = slice(0, 1), slice(1, None)
    return {"first": {key: gather(key, first) for key in ("x", "P")},
            "later": {key: gather(key, later) for key in ("fz", "x", "P", "err_code")}}


def _run_bank(st):
    s, c = st["system"], st["case"]
    _srand(s.srand_seed)
    args = (c["windows"], c["measurements"], s.A0, s.p0, s.b0, s.Phi(0), s.Gamma, np.zeros(0), s.beta, s.H, s.gamma)
    tail = (False, False, False, None, 0.0, 0, np.zeros(0))
    if c["mode"] == "ltv":
        pycauchy.pycauchy_initialize_ltv_window_manager(*args, st["callback"], *tail)
    else:
        pycauchy.pycauchy_initialize_lti_window_manager(*args, *tail)
    try:
        out = [pycauchy.pycauchy_step(z, None) for z in s.zs]
    finally:
        pycauchy.pycauchy_shutdown()
    return {"fz": np.array([o[0] for o in out]), "x": np.array([o[1] for o in out]),
            "P": np.array([o[2] for o in out]), "window": np.array([o[6] for o in out]),
            "err": np.array([o[7] for o in out])}


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "window":
        return _run_window(state)
    if kind == "batch":
        return _run_batch(state)
    if kind == "gradient":
        L = window_loglikelihood(state["theta"], state["systems"])
        (grad,) = torch.autograd.grad(L, state["theta"], state["weight"])
        return {"L": L.detach(), "grad": grad}
    if kind == "orbit":
        L, grad = tangent_gradients(state["systems"], dirs_of=scale_directions)
        return {"L": L, "grad": grad}
    if kind == "bank":
        return _run_bank(state)
    m = case["points"]
    if kind == "relative":
        # the widths are a little over the even division, so that the point count is m
        res = 2.0 / (m - 1) * 1.0001
        out = eval_2d_relative_system_cpdf(state["T"], state["secondary"], state["primary"], 1e-8, -1.0, 1.0, res, -1.0,
                                           1.0, res)
        # out[3:6] are the outputs' own estimates of their rounding errors
        return {"fz": out[0], "x": out[1], "P": out[2], "density": out[6]}
    est, x = state["est"], state["centre"]
    if kind == "marginal1d":
        return list(est.get_marginal_1D_pointwise_cpdf(0, x[0] - 2.0, x[0] + 2.0, 4.0 / (m - 1) * 1.0001))
    j = case["states"] - 1
    res = 2.0 / (m - 1) * 1.0001
    return list(est.get_marginal_2D_pointwise_cpdf(0, j, x[0] - 1.0, x[0] + 1.0, res, x[j] - 1.0, x[j] + 1.0, res))


# ------------------------------------------------------------------------------------ closed forms
def _first_update(A0, p0, b0, H, gamma, z):
    """x = b0 + sum_i A0[i] xi_i with independent Cauchy xi_i of scale p0[i]; z = H x + v with v
    Cauchy of scale gamma: the mean and covariance of x given z."""
    h = A0 @ H
    q = np.abs(h) * p0
    s = q.sum() + gamma
    r = z - H @ b0
    x = b0 + A0.T @ (np.sign(h) * p0) * (r / s)
    D = np.sign(h) * p0
    C = np.diag(p0 * p0 * s / q) - np.outer(D, D)
    P = A0.T @ C @ A0 * (1.0 + (r / s) ** 2)
    return x, P


def exact(case, seed):
    """The first update of a window is closed-form.  The later updates sum millions of terms of
    a tree, the densities are sums over its leaves, and the gradients are their derivatives:
    none has a short form."""
    if case["kind"] == "window":
        if case["mode"] == "nonlin":
            s = W.pendulum_system(p=case["rows"], steps=case["steps"], seed_offset=seed)
            H, z, shift = s.H(s.xbar0)[0], s.zs[0, 0] - s.h(s.xbar0)[0], s.xbar0
        else:
            s = _system(case, seed, case["steps"])
            H, z, shift = s.H[0], s.zs[0, 0], 0.0
        x, P = _first_update(s.A0, s.p0, s.b0, H, s.gamma[0], z)
        return {"first": {"x": x + shift, "P": P}, "later": {"x": None, "P": None, "fz": None, "err": None}}
    if case["kind"] == "batch":
        rows = [_first_update(s.A0, s.p0, s.b0, s.H[0], s.gamma[0], s.zs[0, 0])
                for s in _batch_systems(case["estimators"], seed)]
        return {"first": {"x": np.concatenate([r[0] for r in rows]),
                          "P": np.concatenate([r[1].reshape(-1) for r in rows])},
                "later": {"fz": None, "x": None, "P": None, "err_code": None}}
    return None


# ------------------------------------------------------------------------------------ work
def _terms(n, noises, updates, growth=None):
    g = GROWTH[(n, noises)] if growth is None else growth
    return [(n + 1) * g ** k for k in range(updates)]


def _window_work(n, noises, rows, steps, directions=0, growth=None):
    """Every update writes each term it generates once (m rows of A, p and q, b, c, d in 64 bits)
    and reads it once for its moments and the reduction; a term's g-table is a few dozen cells of
    24 bytes.  About 2000 operations a term: its rows, the moments' product and the cells' two
    complex quotients.  Every tangent direction is as much again."""
    nbytes = flops = 0.0
    for k, terms in enumerate(_terms(n, noises, rows * steps, growth)):
        m = n + noises * (k // rows)
        nbytes += terms * (2 * 8 * (m * (n + 2) + n + 2) + 24 * 2 * m)
        flops += terms * (12 * m * n + 60 * 2 * m)
    return nbytes * (1 + directions), flops * (1 + directions)


def work(case):
    kind = case["kind"]
    if kind == "window":
        b, f = _window_work(case["states"], case["noises"], case["rows"], case["steps"])
    elif kind == "batch":
        every = [_window_work(2 + j % 4, 1, 1, 4 + j // 4 % 5) for j in range(case["estimators"])]
        b, f = (sum(e[i] for e in every) for i in (0, 1))
    elif kind == "gradient":
        b, f = (case["sequences"] * v for v in _window_work(3, 1, 1, case["steps"], 14))
    elif kind == "orbit":
        b, f = (case["windows"] * v for v in _window_work(7, 1, 2, case["steps"], 3, ORBIT_GROWTH))
    elif kind == "bank":
        # each measurement takes one step of every window under way
        b = f = 0.0
        for k in range(case["measurements"]):
            full = _window_work(case["states"], case["noises"], case["rows"], min(k + 1, case["windows"]))
            b, f = b + full[0], f + full[1]
    else:
        n, noises = case["states"], case["noises"]
        updates = case["rows"] * case["steps"]
        # terms that a reduction leaves: about one in ten
        terms = max(1.0, _terms(n, noises, updates + 1)[-1] / 10)
        m = n + noises * case["steps"]
        points = case["points"]
        if kind == "marginal1d":
            b, f = terms * 8 * (m * n + m + n) + 16 * points, terms * points * 8.0
        elif kind == "marginal2d":
            b, f = terms * (8 * (m * n + m + n) + 48 * m) + 24 * points ** 2, terms * points ** 2 * m * 30.0
        else:
            b = 2 * terms * (8 * (m * n + m + n) + 48 * m) + 24 * points ** 2
            f = terms ** 2 * (2 * m * (2 * n + 40) + points ** 2 * 2 * m * 30.0)
    return {"bytes": float(b), "flops": float(f)}
