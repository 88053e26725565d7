"""AsyncProgram on graphs without width: paths, alone and many at once, and a
grid. Levels are exact, and a path alone takes no longer than 64 of them."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def paths(count, length):
    row_ptr = np.tile(np.concatenate([np.arange(length), [length - 1]]), count)
    return (np.full(count, length, np.uint32), np.full(count, length - 1, np.uint64), row_ptr.astype(np.int32),
            np.tile(np.arange(1, length), count).astype(np.int32))


def grid(n):
    i = np.arange(n * n).reshape(n, n)
    a = np.concatenate([i[:, :-1].ravel(), i[:-1].ravel()])
    b = np.concatenate([i[:, 1:].ravel(), i[1:].ravel()])
    src, dst = np.concatenate([a, b]), np.concatenate([b, a])
    order = np.argsort(src, kind="stable")
    row_ptr = np.searchsorted(src[order], np.arange(n * n + 1))
    return (np.array([n * n], np.uint32), np.array([len(dst)], np.uint64), row_ptr.astype(np.int32),
            dst[order].astype(np.int32))


def best_ms(graphs):
    import harmonize_amd as hz

    batch = hz.BfsBatch.from_csr(*graphs)
    want = O.bfs_levels(*graphs)
    ms = []
    for _ in range(5):
        ms.append(batch.run("async", max_launches=1 << 16)["elapsed_ms"])
        assert (batch.levels() == want).all()
    batch.close()
    return min(ms)


def test_one_lane_takes_no_longer_than_sixty_four():
    # Each step is the same trips to memory for one lane as for 64; a quarter
    # of it is left to noise. (One lane took half as long again.)
    assert best_ms(paths(1, 2000)) < 1.25 * best_ms(paths(64, 2000))


@pytest.mark.parametrize("graphs", [paths(3, 2), paths(65, 40), grid(2), grid(90)])
def test_levels(graphs):
    best_ms(graphs)
