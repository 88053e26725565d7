"""Completion words of the resident program's jobs: jobs in flight together
never share one, also where large jobs claimed last are overtaken by more
entries than the doorbell ring holds (the benchmark's burst of 400 jobs, on the
host). Ring positions as words, planted in the oracle, are found."""

import ctypes

import numpy as np
import oracle_lib as O


def shared(sizes, ring):
    f = O.lib().oracle_shared_completion_words
    f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_void_p] + [ctypes.c_uint32] * 3
    sizes = np.ascontiguousarray(sizes, dtype=np.uint32)
    return f(sizes.ctypes.data, len(sizes), 64, ring)


BURST = np.rint(2.0 ** np.random.default_rng(1).uniform(10.0, 22.0, size=400))


def test_jobs_in_flight_have_words_of_their_own():
    assert shared(BURST, 0) == 0
    assert shared(np.concatenate([[1 << 20], np.ones(600), [1 << 20]]), 0) == 0


def test_ring_positions_are_shared():
    assert shared(BURST, 256) > 0
