"""Level hints of the batched search at the sizes where they can go wrong:
levels on both sides of the largest hint, jobs that begin in the middle of a
byte of hints, and visits that overflow a segment of EventProgram's queue."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def path(n):
    """0 - 1 - ... - n-1, both ways: levels up to n - 1, every edge looked at from both ends."""
    return n, [(i, i + 1) for i in range(n - 1)] + [(i + 1, i) for i in range(n - 1)]


def comb(n, tooth):
    """A path whose every vertex has `tooth` leaves, with edges back."""
    edges = list(path(n)[1])
    for i in range(n):
        for k in range(tooth):
            leaf = n + i * tooth + k
            edges += [(i, leaf), (leaf, i)]
    return n + n * tooth, edges


def csr(graph):
    n, edges = graph
    edges = sorted(edges)
    row = np.zeros(n + 1, np.int32)
    for a, _ in edges:
        row[a + 1] += 1
    return np.cumsum(row).astype(np.int32), np.array([b for _, b in edges], np.int32)


@pytest.mark.parametrize("kind,cfg", [("async", {}), ("async", {"block_groups": 4, "stash": 8, "groups": 256}),
                                      ("event", {}), ("event", {"arena": 1 << 13})])
def test_levels_around_the_largest_hint(kind, cfg):
    import harmonize_amd as hz

    graphs = [path(1), path(14), path(15), path(16), path(17), comb(33, 129), path(3), comb(5, 1), path(64)]
    v, e, rows, cols = [], [], [], []
    for g in graphs:
        r, c = csr(g)
        v.append(g[0])
        e.append(len(c))
        rows.append(r)
        cols.append(c)
    v, e = np.array(v, np.uint32), np.array(e, np.uint64)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    want = O.bfs_levels(v, e, rows, cols)
    assert want.max() == 63 and (want == 14).any() and (want == 15).any()
    b = hz.BfsBatch.from_csr(v, e, rows, cols)
    for _ in range(2):  # a second search starts from fresh hints
        b.run(kind, max_launches=1 << 16, **cfg)
        assert np.array_equal(b.levels(), want)
    b.close()
