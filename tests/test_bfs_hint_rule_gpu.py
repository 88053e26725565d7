"""Where a batch is searched through level hints: only where they are faster,
with the same levels either way, and by turns on one batch."""

import numpy as np
import pytest

import oracle_lib as O
from test_bfs_hints_gpu import comb, csr, path

pytestmark = pytest.mark.gpu

GRAPH, AUDIT, HINTS = 1, 2, 4  # HZ_RUN_GRAPH, HZ_RUN_AUDIT, HZ_RUN_LEVEL_HINTS


def ring(n, degree, width):
    """Each vertex has neighbours within `width` places: far more than 14 levels."""
    r = np.random.default_rng(1)
    col = (np.repeat(np.arange(n), degree) + r.integers(-width, width + 1, n * degree)) % n
    return (np.array([n], np.uint32), np.array([n * degree], np.uint64),
            np.arange(0, n * degree + 1, degree, dtype=np.int32), col.astype(np.int32))


def test_a_deep_search_does_not_pay_for_hints():
    import harmonize_amd as hz

    graph = ring(1 << 19, 32, 500)
    batch = hz.BfsBatch.from_csr(*graph)
    want = O.bfs_levels(*graph)
    best = {}
    for _ in range(7):
        for flags in (0, HINTS):
            ms = batch.run("async", flags=flags, max_launches=1 << 16)["elapsed_ms"]
            best[flags] = min(ms, best.get(flags, ms))
            assert np.array_equal(batch.levels(), want)
    batch.close()
    # 14.7 against 17.7 ms; a third of the difference is enough.
    assert best[0] < 0.95 * best[HINTS]


@pytest.mark.parametrize("kind,cfg", [("async", {}), ("async", {"block_groups": 2}),
                                      ("async", {"block_groups": 4, "stash": 8, "groups": 256}),
                                      ("async", {"flags": GRAPH}), ("async", {"flags": AUDIT}),
                                      ("event", {}), ("event", {"arena": 1 << 13})])
def test_same_levels_by_turns(kind, cfg):
    import harmonize_amd as hz

    graphs = [path(1), path(14), path(15), path(16), path(17), comb(33, 129), path(3), comb(5, 1), path(64)]
    rows, cols = zip(*(csr(g) for g in graphs))
    v = np.array([g[0] for g in graphs], np.uint32)
    e = np.array([len(c) for c in cols], np.uint64)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    want = O.bfs_levels(v, e, rows, cols)
    batch = hz.BfsBatch.from_csr(v, e, rows, cols)
    for hints in (0, HINTS, HINTS, 0, HINTS):
        batch.run(kind, max_launches=1 << 16, **{**cfg, "flags": cfg.get("flags", 0) | hints})
        assert np.array_equal(batch.levels(), want)
    batch.close()


@pytest.mark.parametrize("edge_factor", [15, 16, 32])
def test_both_sides_of_the_rule(edge_factor):
    # 2^28 edges and more are searched through hints by EventProgram, 2^29 by both.
    import harmonize_amd as hz

    batch = hz.BfsBatch.rmat(3, np.full(16, 1 << 20, np.uint32), edge_factor)
    levels = []
    for kind, flags in (("event", 0), ("async", 0), ("event", HINTS), ("async", HINTS)):
        batch.run(kind, flags=flags, max_launches=1 << 16)
        levels.append(batch.levels())
    batch.close()
    for other in levels[1:]:
        assert np.array_equal(levels[0], other)
