"""Generations of EventProgram that grow late: a search that follows a path, and
so has been given few groups, into a graph of millions. Levels are exact, a
bound on launches counts generations as before, and the search costs the
generations of the path beside that of the graph alone."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

VERTICES = 1 << 21


@pytest.fixture(scope="module")
def hz():
    import harmonize_amd

    return harmonize_amd


def behind_a_path(hz, length, seed=9, vertices=VERTICES):
    """A batch of one R-MAT graph that is entered through a path of `length` vertices."""
    b = hz.BfsBatch.rmat(seed, np.array([vertices], np.uint32))
    row_ptr, col = b.csr()
    b.close()
    row_ptr = np.concatenate([np.arange(length), length + row_ptr]).astype(np.int32)
    col = np.concatenate([np.arange(1, length + 1), col + length]).astype(np.int32)
    v, e = np.array([vertices + length], np.uint32), np.array([len(col)], np.uint64)
    return hz.BfsBatch.from_csr(v, e, row_ptr, col), O.bfs_levels(v, e, row_ptr, col)


def best_ms(hz, batch, want):
    ms = []
    for _ in range(5):
        ms.append(batch.run("event", max_launches=1 << 16)["elapsed_ms"])
        assert (batch.levels() == want).all()
    return min(ms)


def test_late_growth_gets_its_groups(hz):
    short, want_short = behind_a_path(hz, 1)
    long, want_long = behind_a_path(hz, 40)
    # 39 generations more of 50 us at most (10 on the device, looks, and one
    # batch of launches that leave a grown generation to the next): 2 ms, and
    # as much again for noise. On 66 groups the graph alone takes 15 ms more.
    assert best_ms(hz, long, want_long) < best_ms(hz, short, want_short) + 4.0
    short.close()
    long.close()


@pytest.mark.parametrize("length", [16, 17, 31, 33])
@pytest.mark.parametrize("groups", [0, 70])
def test_launch_bounds_count_generations(hz, length, groups):
    batch, want = behind_a_path(hz, length, vertices=1 << 16)
    n = batch.run("event", max_launches=1 << 16, groups=groups)["launches"]
    assert (batch.levels() == want).all()
    assert batch.run("event", max_launches=n, groups=groups)["launches"] == n
    with pytest.raises(hz.HarmonizeError, match="launch bound"):
        batch.run("event", max_launches=n - 1, groups=groups)
    batch.close()
