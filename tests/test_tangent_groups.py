"""Tangents of the reduction groups' g-tables on both sides of the number of groups beyond
which one wavefront takes a group instead of four."""
import numpy as np
import pytest

from cauchyfriendly_amd import workloads as W


# 7-state orbit windows: at 3 steps every update has fewer than 4096 groups, at 4 the largest more.
@pytest.mark.gpu
@pytest.mark.parametrize("steps", [3, 4])
def test_scale_tangents_match_central_differences(steps):
    from cauchyfriendly_amd.likelihood import scale_directions, scale_gradient, tangent_gradients
    ws = W.leo7_windows(2, steps, dt=1.0, seed_offset=4)
    L, grad = tangent_gradients(ws, dirs_of=scale_directions)
    d = scale_gradient(ws, h=1e-6, num_threads=2, max_live=4, details=True)
    assert d["valid"].any()
    for i in range(len(ws)):
        assert abs(float(L[i]) - d["L"][i]) <= 1e-12 * abs(d["L"][i])
        for j in range(d["h"].shape[1]):
            if not d["valid"][i, j]:
                continue
            # a difference's round-off (1e-12 relative per likelihood over 2h) and 1e-5 of it
            tol = 1e-12 * abs(d["L"][i]) / d["h"][i, j] + 1e-5 * max(1.0, abs(d["grad"][i, j]))
            print(f"  window {i} scale {j}: {float(grad[i][j])} {d['grad'][i, j]}", flush=True)
            assert abs(float(grad[i][j]) - d["grad"][i, j]) <= tol
