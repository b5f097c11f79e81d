"""Host threads that come and go: each takes over the streams, staging memory and device
blocks of those that ended, and steps its window to the same bits."""
import threading

import numpy as np
import pytest

from cauchyfriendly_amd import workloads as W
from cauchyfriendly_amd.estimator import run_system


def _window(s, steps):
    out = run_system(s, num_steps=steps)[1]
    return [np.concatenate([np.ravel(u[key]) for key in ("fz", "mean", "cov")]).tobytes() for u in out]


@pytest.mark.gpu
@pytest.mark.parametrize("threads", [1, 5])
def test_windows_of_fresh_threads_keep_their_bits(threads):
    # the last update of the 5-state window takes blocks beyond the power-of-two classes
    s = W.config1(steps=5)
    want = _window(s, 5)
    for _ in range(3):
        got = [None] * threads

        def run(i):
            got[i] = _window(s, 5)

        ts = [threading.Thread(target=run, args=(i,)) for i in range(threads)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert all(g == want for g in got)
