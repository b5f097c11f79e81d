"""Reduction groups' g-tables where the lookup changes: every mode with every member evaluated
by a wavefront of its own, and the largest shape on both sides of the 16 rows up to which a
parent's table is looked up by rank."""
import numpy as np
import pytest

from conftest import compare_update, load_golden
from cauchyfriendly_amd import workloads as W
from cauchyfriendly_amd.estimator import GpuEstimator

pytestmark = pytest.mark.gpu


def _run(s, window, steps):
    est = GpuEstimator(window, s.n, s.pncc, s.p, s.A0, s.p0, s.b0, cmcc=s.cmcc, seed=s.srand_seed)
    G = np.ascontiguousarray(s.Gamma.reshape(-1))
    B = None if s.B is None else np.ascontiguousarray(s.B.reshape(-1))
    out = [est.step(s.zs[k, i], s.Phi(k).reshape(-1), G, s.beta, s.H[i], s.gamma[i], B, s.u(k))
           for k in range(steps) for i in range(s.p)]
    est.close()
    return out


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
def test_members_of_their_own_wavefronts_in_every_mode(mode, monkeypatch):
    monkeypatch.setenv("MCE_GEVAL_MODE", str(mode))
    monkeypatch.setenv("MCE_BIG_GROUP_MEMBERS", "0")
    rec = load_golden("lti3_w8")
    s = W.System.from_dict(rec["system"])
    print(f"case mode {mode}", flush=True)
    for u, (got, exp) in enumerate(zip(_run(s, rec["num_steps"], rec["num_steps"]), rec["updates"])):
        compare_update(got, exp, 1e-9, where=f"mode {mode} update {u}")


def test_results_are_alike_on_both_sides_of_sixteen_rows():
    # a window of n steps of a 2-state, one-noise system has n + 1 rows; the largest shape
    # bounds the tables, not the terms, so the first updates are the same
    s = W.lti_system(d=2, steps=19, seed_offset=5)
    runs = []
    for window in (15, 16, 19):
        print(f"case window {window}: {window + 1} rows", flush=True)
        runs.append(_run(s, window, 8))
    for other in runs[1:]:
        for a, b in zip(runs[0], other):
            assert a["nt_mu"] == b["nt_mu"] and a["nt_ftr"] == b["nt_ftr"]
            for key in ("fz", "mean", "cov"):
                assert np.array_equal(np.asarray(a[key]), np.asarray(b[key])), key
