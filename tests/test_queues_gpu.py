"""Links that travel between groups through the device queues: batches of
free links, the count of holders, and searches whose links spill, are handed
to waiting groups and resumed by later launches. Levels are exact and every
launch is audited (no link lost, queued twice or left out of the counts)."""

import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

SEED = 0xB0FF


@pytest.fixture(scope="module")
def batch():
    import harmonize_amd as hz

    b = hz.BfsBatch.rmat(SEED, hz.bfs_batch_sizes(SEED, 9, 5.0, 15.0))
    row_ptr, col = b.csr()
    yield hz, b, O.bfs_levels(b.vertices, b.edges, row_ptr, col)
    b.close()


# arena / (16 x groups) is the batch of links a group claims and gives back:
# below 2, at 2, between, and beyond the 16 that a group handles at a time.
@pytest.mark.parametrize("groups,arena", [(64, 1 << 12), (48, 1536), (64, 1 << 13), (16, 1 << 14), (333, 1 << 18)])
@pytest.mark.parametrize("queues,cycles", [(1, 0), (3, 40), (64, 7)])
def test_links_through_the_queues(batch, groups, arena, queues, cycles):
    hz, b, want = batch
    st = b.run("async", groups=groups, arena=arena, queues=queues, cycles=cycles, stash=8, spec_param=16,
               max_launches=1 << 20, flags=hz.RUN_AUDIT)
    assert (b.levels() == want).all()
    assert st["audits"] == st["launches"]
