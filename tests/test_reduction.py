"""Fast term reduction by components of one sort key (k_ftr_keys, k_ftr_comp, k_ftr_comp_big)."""
import ctypes as ct

import numpy as np
import pytest

from conftest import rel_err
from cauchyfriendly_amd import pycauchy
from cauchyfriendly_amd import workloads as W
from cauchyfriendly_amd.estimator import run_system

EPS = 1e-8
RING = 2 ** 34
_dp, _ip = ct.POINTER(ct.c_double), ct.POINTER(ct.c_int)


def _lib():
    from cauchyfriendly_amd import _native
    L = _native.lib()
    L.mce_reduction_key.restype = L.mce_reduction_link.restype = ct.c_uint64
    L.mce_reduction_key.argtypes = [ct.c_int, ct.c_int, _dp, _dp, _dp]
    L.mce_reduce_terms.argtypes = [ct.c_void_p, ct.c_int, _ip, _dp, _dp, _dp, _ip, _ip]
    return L


def _c(a):
    return a.ctypes.data_as(_ip if a.dtype == np.int32 else _dp)


def _key(b, p, A):
    """The sort key of one term as the reduction forms it, without the shape bits."""
    b, p, A = (np.ascontiguousarray(v, dtype=np.float64) for v in (b, p, A))
    k = _lib().mce_reduction_key(len(b), len(p), _c(b), _c(p), _c(A))
    assert k >> 34 == len(p)
    return k % RING


@pytest.mark.parametrize("d,m", [(1, 1), (2, 20), (3, 14), (5, 15), (8, 12)])
@pytest.mark.parametrize("scale", [1e-3, 1.0, 1e3, 1e6, 1e7, 1e8, 1e9, 1e12])
def test_terms_within_the_tolerances_are_linked(d, m, scale):
    """Two terms that the reduction's comparisons accept never have keys further apart than the
    distance at which sorted neighbours are linked, also at the edge of every comparison and where
    it is a rounding of the last place."""
    rng = np.random.default_rng(20261202 + 100 * d + m)
    link = _lib().mce_reduction_link(d, m)
    for _ in range(200):
        b, p = (scale * rng.standard_cauchy(n) for n in (d, m))
        b = np.where(rng.random(d) < 0.2, 2.0 ** rng.integers(24, 30, d) * rng.choice([-1, 1], d), b)
        A = rng.uniform(-1, 1, m)
        # the ends of b's window (b - EPS, b + EPS], of p's interval, and A within it up to its sign
        b2 = np.where(rng.random(d) < 0.5, b + EPS, np.nextafter(b - EPS, np.inf))
        b2 = np.where((b2 > b - EPS) & (b2 <= b + EPS), b2, b)
        p2 = p + EPS * rng.choice([-1, 1], m)
        p2 = np.where(np.abs(p2 - p) > EPS, np.nextafter(p2, p), p2)
        p2 = np.where(np.abs(p2 - p) > EPS, p, p2)
        A2 = rng.choice([-1, 1], m) * (A + 0.999 * EPS * rng.choice([-1, 1], m))
        gap = (_key(b, p, A) - _key(b2, p2, A2)) % RING
        assert min(gap, RING - gap) <= link


# for each system up to the largest unit in which rounding leaves the reduction as it is in units of one
@pytest.mark.parametrize("d,steps,seed,scale", [
    (d, steps, seed, u) for d, steps, seed, most in [(2, 7, 5, 1e6), (2, 7, 7, 1e5), (3, 6, 125, 1e4)]
    for u in (1e-3, 1.0, 1e4, 1e5, 1e6) if u <= most])
def test_terms_that_do_not_reduce_are_told_apart_in_any_unit(d, steps, seed, scale):
    """Sorted runs of linked keys among terms that do not reduce, in states of any unit, end within
    the 64 positions that one wavefront looks at."""
    from oracle import driver as dr
    s = W.ltv_system(d=d, steps=steps, seed_offset=seed, pncc=2, p=1, beta=0.05 * scale, gamma=0.1 * scale,
                     p0=0.1 * scale)
    _, recs = dr.run_system(s, kind="oracle", collect_terms=True)
    terms = recs[-2]["terms"]
    longest = {}
    for m in sorted({t["m"] for t in terms}):
        link = _lib().mce_reduction_link(d, m)
        keys = np.sort([_key(t["b"], t["p"], t["A"].ravel()[:m]) for t in terms if t["m"] == m])
        runs = np.split(keys, 1 + np.flatnonzero(np.diff(keys) > link))
        longest[m] = max(len(r) for r in runs)
    print(f"  {len(terms)} terms, longest runs by shape {longest}")
    assert len(terms) > 1000 and max(longest.values()) < 64


def _given(d, MM, shape, b, p, A):
    """Root and place of each term by the reduction's kernels, and by the restatement."""
    from cauchyfriendly_amd.estimator import GpuEstimator
    from oracle import driver as dr
    n = len(shape)
    shape = np.asarray(shape, dtype=np.int32)
    b, p, A = (np.ascontiguousarray(v, dtype=np.float64) for v in (b, p, A))
    root, place = np.full(n, -2, dtype=np.int32), np.full(n, -2, dtype=np.int32)
    est = GpuEstimator(MM - d + 1, d, 1, 1, np.eye(d), np.ones(d), np.zeros(d), seed=1)
    L = _lib()
    assert L.mce_shape_range(est.h) == MM + 1
    rc = L.mce_reduce_terms(est.h, n, _c(shape), _c(b), _c(p), _c(A), _c(root), _c(place))
    assert rc == 0, L.mce_last_error()
    est.close()
    want = np.empty(n, dtype=np.int32)
    for m in np.unique(shape):
        at = np.flatnonzero(shape == m)
        F = np.empty(len(at), dtype=np.int32)
        bm, pm, Am = (np.ascontiguousarray(v[at]) for v in (b, p[:, :m], A[:, :m]))
        dr.lib("oracle")._cdll.oracle_reduce(len(at), d, int(m), _c(bm), _c(pm), _c(Am), _c(F))
        want[at] = at[F]
    order = np.full(n, -1, dtype=np.int32)
    for r in np.unique(want):
        mem = np.flatnonzero((want == r) & (np.arange(n) != r))
        order[mem] = np.arange(len(mem))
    return root, place, want, order


def _across_zero(rng, d, m, n, spread):
    """n terms around a key of zero, `spread` key units to either side: the run that a shape's last
    keys begin and its first ones go on."""
    b, p, A = rng.uniform(-1, 1, d), rng.uniform(0, 1, m), rng.uniform(-1, 1, m)
    lo, hi = 0.0, 2.0 ** 10  # b[0]'s weight lies in [1/2, 1): the key crosses zero on the way
    at = lambda x: _key(np.r_[x, b[1:]], p, A)
    k0 = at(0.0)
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        if (at(mid) - k0) % RING < (RING - k0) % RING and mid < 256:
            lo = mid
        else:
            hi = mid
    bs = np.tile(np.r_[hi, b[1:]], (n, 1))
    bs[:, 0] += spread * 2.0 ** -26 * rng.uniform(-1, 1, n)
    return bs, np.tile(p, (n, 1)), np.tile(A, (n, 1))


GIVEN = ["alike", "noise", "near", "across_few", "across_many", "across_chunks", "shapes", "nan", "huge"]


@pytest.mark.gpu
@pytest.mark.parametrize("case", GIVEN)
def test_given_terms_reduce_like_the_restatement(case):
    rng = np.random.default_rng(20261205 + GIVEN.index(case))
    d, MM, m = 2, 8, 5
    if case == "alike":  # one group of thousands, and in a bucket reduced in 8 chunks
        n = 10007
        b, p, A = np.tile([0.3, -2.0], (n, 1)), np.tile(rng.uniform(0, 1, m), (n, 1)), np.tile(rng.uniform(-1, 1, m), (n, 1))
        A *= rng.choice([-1, 1], (n, m))
    elif case == "noise":  # 40 groups of 300, keys not equal
        n = 12000
        c = rng.integers(0, 40, n)
        b = (1e4 * rng.standard_normal((40, d)))[c] + 1e-10 * rng.standard_normal((n, d))
        p, A = rng.uniform(0, 1, (40, m))[c], rng.uniform(-1, 1, (40, m))[c]
    elif case == "near":  # nearly every term its own root, keys without gaps
        n = 3000
        b, p, A = 1e-6 * rng.standard_normal((n, d)), 1e-6 * rng.uniform(0, 1, (n, m)), np.full((n, m), 0.25)
    elif case in ("across_few", "across_many", "across_chunks"):
        n = {"across_few": 20, "across_many": 1500, "across_chunks": 10500}[case]
        b, p, A = _across_zero(rng, d, m, n, {"across_few": 2.0, "across_many": 40.0, "across_chunks": 300.0}[case])
        far = 200  # other terms of the shape on both sides
        b, p, A = (np.vstack([v, rng.uniform(-3, 3, (far, v.shape[1]))]) for v in (b, p, A))
        mix = rng.permutation(n + far)
        b, p, A = b[mix], p[mix], A[mix]
        keys = np.array([_key(*t) for t in zip(b[:2000], p, A)])
        assert (keys < RING // 8).any() and (keys > RING - RING // 8).any()
    elif case == "nan":  # a NaN in p compares as equal to anything
        n = 400
        c = rng.integers(0, 20, n)
        b, p, A = rng.uniform(-1, 1, (20, d))[c], rng.uniform(0, 1, (20, m))[c], rng.uniform(-1, 1, (20, m))[c]
        p[rng.random((n, m)) < 0.02] = np.nan
        p[rng.random((n, m)) < 0.02] = np.inf
    elif case == "huge":  # magnitudes at which the tolerance is below the last place
        n = 4000
        c = rng.integers(0, 1000, n)
        b = (2.0 ** rng.uniform(20, 40, (1000, d)) * rng.choice([-1, 1], (1000, d)))[c] + 1.5e-8 * rng.integers(0, 2, (n, d))
        p, A = (2.0 ** rng.uniform(20, 40, (1000, m)))[c], rng.uniform(-1, 1, (1000, m))[c]
        p[0, 0], b[1, 1] = np.inf, -np.inf
    if case == "shapes":  # small buckets side by side, some across zero
        rows = []
        for k in range(1, MM + 1):
            bb, pp, AA = _across_zero(rng, d, k, 5 * k, 3.0)
            pad = np.zeros((5 * k, MM - k))
            rows.append((np.full(5 * k, k), bb, np.hstack([pp, pad]), np.hstack([AA, pad])))
        shape, b, p, A = (np.concatenate(v) for v in zip(*rows))
    else:
        shape = np.full(len(b), m)
        pad = np.zeros((len(b), MM - m))
        p, A = np.hstack([p, pad]), np.hstack([A, pad])
    print(f"case {case}: {len(b)} terms", flush=True)
    root, place, want, order = _given(d, MM, shape, b, p, A)
    print(f"  {len(np.unique(want))} roots", flush=True)
    assert np.array_equal(root, want)
    assert np.array_equal(place, order)


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


# Units in which the keys have no gaps at one end, and in which nothing but equal numbers reduces
# at the other.
@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-5, 1e-4, 1e4, 1e6])
def test_units_do_not_change_what_reduces(scale):
    print(f"case scale {scale}", flush=True)
    s = W.ltv_system(d=2, steps=8, seed_offset=5, pncc=2, p=1, beta=0.05 * scale, gamma=0.1 * scale, p0=0.1 * scale)
    _same_as_the_restatement(s, 8)


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
