"""Workspaces that a finished run leaves for the next one: calls of several
threads at once, of alternating sizes and kinds, after a call that failed, and
after the idle workspaces were freed, all equal the oracle."""

import threading

import numpy as np
import pytest

import harmonize_amd as hz
import oracle_lib as O

pytestmark = pytest.mark.gpu


def collatz(seed, n, kind="async", **cfg):
    host = O.collatz_make_starts(seed, 40, n)
    steps = hz.DeviceArray(n, np.uint32)
    st = hz.collatz_run(kind, steps, hz.DeviceArray.from_numpy(host), max_launches=100000, **cfg)
    ref, promises = O.collatz_steps(host)
    assert np.array_equal(steps.numpy(), ref)
    assert st["promises"] == promises


def test_threads_have_a_workspace_each():
    failed = []

    def work(t):
        try:
            for i in range(6):
                collatz(100 * t + i, 1000 + 517 * ((t + i) % 3), "event" if (t + i) % 4 == 3 else "async")
        except BaseException as e:  # reported by the test's own thread
            failed.append(e)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


def test_sizes_alternate_and_release():
    for i in range(4):
        collatz(i, 3000, arena=1 << (10 + i % 2), queues=1 + i % 3)
        if i % 2 == 1:
            hz.workspace_release()
    total, echo, forwarded, _ = hz.futures_run("async", hz.DeviceArray.from_numpy(np.arange(1, 65, dtype=np.uint64)), 5)
    again = hz.futures_run("async", hz.DeviceArray.from_numpy(np.arange(1, 65, dtype=np.uint64)), 5)
    assert total == again[0] and np.array_equal(echo, again[1]) and np.array_equal(forwarded, again[2])


def test_a_failed_run_leaves_nothing_behind():
    n = 1 << 16
    steps = hz.DeviceArray(n, np.uint32)
    for _ in range(2):
        with pytest.raises(hz.HarmonizeError, match="arena"):
            hz.collatz_run("async", steps, None, n, cycles=50, groups=256, arena=4, max_launches=1000)
    collatz(5, 20000, cycles=50, groups=256, arena=4096)
