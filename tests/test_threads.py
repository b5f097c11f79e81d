"""Host threads that come and go: each takes over the streams, staging memory and device
blocks of those that ended, and steps its window to the same bits."""
import ctypes as ct
import threading
import time

import numpy as np
import pytest

from cauchyfriendly_amd import _native
from cauchyfriendly_amd import workloads as W
from cauchyfriendly_amd.estimator import run_system, trim_device_memory


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


def _free_bytes():
    free, total = ct.c_size_t(), ct.c_size_t()
    # by way of the engine's handle: the runtime that the engine itself uses
    assert _native.lib().hipMemGetInfo(ct.byref(free), ct.byref(total)) == 0
    return free.value


def _large_window():
    est, _ = run_system(W.config1(steps=5), num_steps=5)
    est.close()


@pytest.mark.gpu
def test_idle_blocks_go_back_to_the_device():
    run_system(W.config0())[0].close()  # slabs stay with the process
    trim_device_memory()
    before = _free_bytes()
    _large_window()
    kept = before - _free_bytes()
    print(f"kept {kept >> 20} MiB", flush=True)
    assert kept > 256 << 20
    freed = trim_device_memory()
    slabs = before - _free_bytes()
    # the runtime cuts blocks of a few MiB from chunks of its own: 64 MiB either way
    assert freed > 256 << 20 and abs(kept - freed - slabs) <= 64 << 20
    # large blocks go once they lay unused for 10 s and any estimator takes or gives back a block
    _large_window()
    time.sleep(10.5)
    print("10.5 s later", flush=True)
    run_system(W.config0())[0].close()
    # what is left: slabs and the blocks of up to 256 MiB
    left = before - _free_bytes()
    assert left <= kept - (256 << 20)
    assert trim_device_memory() <= left + (64 << 20)
