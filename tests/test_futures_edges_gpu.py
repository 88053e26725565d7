"""Futures trees at the sizes where lanes that chain change hands: fewer
leaves than lanes, a link's edges, chains of one step and of hundreds side by
side, joins too few to fill a link, and launches cut short with chains and
held readers in flight. Bit-exact against the host executors."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaves,readers", [(1, 1), (2, 0), (32, 65), (64, 1), (128, 63), (4096, 64)])
@pytest.mark.parametrize("what", ["short", "mixed", "long"])
@pytest.mark.parametrize("cfg", [{}, {"groups": 3, "cycles": 24}, {"groups": 700, "queues": 1}])
def test_tree_edges(leaves, readers, what, cfg):
    import harmonize_amd as hz

    i = np.arange(leaves, dtype=np.uint64)
    starts = {"short": i % 3, "mixed": np.where(i % 5 == 0, np.uint64(837799), i % 2), "long": 837799 + 0 * i}[what]
    dev = hz.DeviceArray.from_numpy(np.ascontiguousarray(starts, dtype=np.uint64))
    total, echo, forwarded, st = hz.futures_run("async", dev, readers, max_launches=1 << 20, flags=hz.RUN_AUDIT, **cfg)
    ref_total, ref_echo, ref_forwarded, ref = O.futures_program(dev.numpy(), readers, threads=0)
    assert total == ref_total and st["promises"] == ref.promises
    assert np.array_equal(echo, ref_echo) and np.array_equal(forwarded, ref_forwarded)
    assert st["audits"] == st["launches"]
