"""Fast term reduction by components of one sort key (k_ftr_keys, k_ftr_comp, k_ftr_comp_big)."""
import ctypes as ct

import numpy as np
import pytest

from conftest import rel_err
from cauchyfriendly_amd import pycauchy
from cauchyfriendly_amd import workloads as W
from cauchyfriendly_amd.estimator import run_system

EPS = 1e-8


def _key(b, p, A):
    """The sort key of one term, as k_ftr_keys forms it (without the shape bits)."""
    d, m = len(b), len(p)
    w = lambda k: 0.5 + 0.5 * np.modf((k + 1) * 0.6180339887498949)[0]
    f = lambda x: min(abs(x), 1e300) / (1.0 + min(abs(x), 1e300))
    v = 128.0 + sum(w(a) * np.copysign(f(b[a]), b[a]) for a in range(d))
    for k in range(m):
        v += w(d + 2 * k) * np.copysign(f(p[k]), p[k]) + w(d + 2 * k + 1) * f(A[k])
    return int(v * 2.0 ** 26)


@pytest.mark.parametrize("d,m,scale", [(1, 1, 1.0), (2, 20, 1e-3), (3, 14, 1.0), (5, 15, 1e3), (8, 12, 1e6)])
def test_terms_within_the_tolerances_are_linked(d, m, scale):
    """Two terms that the reduction's comparisons accept never have keys further apart than the
    distance at which sorted neighbours are linked, also at the edge of every comparison."""
    rng = np.random.default_rng(20261202 + 100 * d + m)
    link = int(0.672 * (d + 2 * m)) + 3
    for _ in range(400):
        b, p, A = (scale * rng.standard_cauchy(n) for n in (d, m, m))
        # a shift of b and p by the tolerance (or what is left of it at these magnitudes) ...
        b2 = b + EPS * rng.choice([-1, 1, 0.999], d)
        p2 = p + EPS * rng.choice([-1, 1], m)
        # ... and A within it up to its sign
        A2 = rng.choice([-1, 1], m) * (A + EPS * rng.uniform(-1, 1, m))
        ka, kb = _key(b, p, A), _key(b2, p2, A2)
        assert 0 <= ka < 2 ** 34 and abs(ka - kb) <= link


def _same_as_the_restatement(s, steps):
    from oracle import driver as dr
    _, g = run_system(s, num_steps=steps)
    o = dr.run_system(s, num_steps=steps, kind="oracle")[1]
    for u, (a, b) in enumerate(zip(g, o)):
        print(f"  update {u}: {a['nt_mu']} -> {a['nt_ftr']}", flush=True)
        assert np.array_equal(a["shape_mu"], b["shape_mu"]) and np.array_equal(a["shape_ftr"], b["shape_ftr"])
        assert a["err"] == b["err"]
        assert max(rel_err(a["fz"], b["fz"]), rel_err(a["mean"], b["mean"]), rel_err(a["cov"], b["cov"])) <= 1e-9


# The 2-state window of 10 steps has components of 458 and 1458 terms in buckets reduced at once
# and of 4398, 5116 and 16269 terms in buckets reduced in 8 chunks; the others end inside one
# wavefront's 64 positions or straddle them.
@pytest.mark.gpu
@pytest.mark.parametrize("d,pncc,steps,seed", [(1, 1, 12, 3), (2, 1, 9, 5), (2, 2, 10, 7), (3, 2, 6, 9), (7, 1, 4, 11)])
def test_components_reduce_like_the_restatement(d, pncc, steps, seed):
    print(f"case d={d} pncc={pncc} steps={steps} seed={seed}", flush=True)
    if pncc == 1:
        s = W.lti_system(d=d, steps=steps, seed_offset=seed)
    else:
        s = W.ltv_system(d=d, steps=steps, seed_offset=seed, pncc=pncc, p=1)
    _same_as_the_restatement(s, steps)


@pytest.mark.gpu
@pytest.mark.parametrize("ordering", [[1, 2, 0], [2, 0, 1]])
def test_any_search_order_reduces_like_the_restatement(ordering):
    from oracle import driver as dr
    o = np.array(ordering, dtype=np.int32)
    identity = np.arange(12, dtype=np.int32)
    ip = ct.POINTER(ct.c_int)
    L = dr.lib("oracle")
    try:
        assert pycauchy.pycauchy_set_tr_search_idxs_ordering(o) == 0
        assert L.ref_set_tr_search_idxs_ordering(o.ctypes.data_as(ip), len(o)) == 0
        _same_as_the_restatement(W.config0(), 8)
    finally:
        pycauchy.pycauchy_set_tr_search_idxs_ordering(identity)
        L.ref_set_tr_search_idxs_ordering(identity.ctypes.data_as(ip), 12)
