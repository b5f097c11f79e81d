"""Tangents of the reduction groups' g-tables: one wavefront per group and four per group form
the same sums in the same order, so the gradients agree to the last bit."""
import numpy as np
import pytest

from cauchyfriendly_amd import workloads as W


# 7-state orbit windows have groups of hundreds of members and of none; the 3-state windows
# have 14 directions, tables below 64 cells and merged hyperplanes; the 5-state ones two noises.
@pytest.mark.gpu
@pytest.mark.parametrize("case", ["orbit", "lti", "ltv"])
def test_wavefronts_per_group_leave_the_gradient_alone(case, monkeypatch):
    from cauchyfriendly_amd.likelihood import scale_directions, tangent_gradients, theta_directions
    if case == "orbit":
        ws, dirs = W.leo7_windows(2, 4, dt=1.0, seed_offset=4), scale_directions
    elif case == "lti":
        ws, dirs = W.lti_sequences(4), theta_directions
    else:
        ws, dirs = [W.ltv_system(d=5, steps=3, seed_offset=1, pncc=2, p=2)], scale_directions
    got = []
    for first in (0, 1 << 30):  # one wavefront from the first group on, or never
        monkeypatch.setenv("MCE_TAN_ONE_WAVE", str(first))
        print(f"case {case}: one wavefront from {first} groups on", flush=True)
        got.append(tangent_gradients(ws, dirs_of=dirs))
    for a, b in zip(*got):
        a, b = np.asarray(a), np.asarray(b)
        assert np.all(np.isfinite(a)) and a.tobytes() == b.tobytes()
