"""Idle memory is given back where an allocation needs it: on a device with less
memory left than a call needs, and idle workspaces that fill the gap, a
server, a batch, a search and a run are still made. Where the gap is filled by
memory in use, the same call is refused, and the next one works."""

import ctypes
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


HOGS = []


@pytest.fixture(scope="module")
def batch():
    import harmonize_amd

    b = harmonize_amd.BfsBatch.rmat(3, np.array([1000], np.uint32))
    warm(harmonize_amd)
    yield b
    b.close()
    HOGS.clear()


@pytest.fixture
def hz(batch):
    """The runtime on a device with 1,000 MiB left."""
    import harmonize_amd

    gc.collect()  # what other tests have left
    harmonize_amd.workspace_release()
    for _ in range(4):  # what is left is not exact right after a large allocation
        free = free_mib()
        if free > 1016:
            HOGS.append(harmonize_amd.DeviceArray((free - 1000) * MIB, np.uint8))
    assert 900 < free_mib() < 1100
    return harmonize_amd


def free_mib():
    import harmonize_amd as hz

    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hz.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value // MIB


def run_idle(hz, kind, arena):
    hz.collatz_run(kind, hz.DeviceArray(64, np.uint32), None, 64, arena=arena, groups=64, max_launches=1000)


def warm(hz):
    run_idle(hz, "async", 64)
    run_idle(hz, "event", 4096)


@pytest.mark.parametrize("what", ["resident", "server", "batch", "search", "run"])
def test_idle_memory_makes_room(hz, batch, what):
    run_idle(hz, "async", 1 << 19)  # 513 MiB and more
    run_idle(hz, "event", 1 << 21)  # 128 MiB
    assert free_mib() < 450
    if what == "resident":
        hz.Resident(pool_bytes=520 * MIB, arena_links=1 << 12).close()
    elif what == "server":
        hz.Server(pool_bytes=8 * MIB, slots=1, arena_links=1 << 12).close()  # 512 MiB of queues
    elif what == "batch":
        hz.BfsBatch.rmat(3, np.array([1 << 21], np.uint32)).close()
    elif what == "search":
        assert batch.run("event", arena=(520 * MIB) // 64)["promises"] > 0
    else:
        st = hz.collatz_run("async", hz.DeviceArray(64, np.uint32), None, 64, arena=480 << 10, groups=64)
        assert st["promises"] > 0


def test_memory_in_use_is_refused(hz):
    used = hz.DeviceArray(640 * MIB, np.uint8)
    with pytest.raises(hz.HarmonizeError, match="out of memory"):
        hz.Resident(pool_bytes=900 * MIB)
    warm(hz)
    used.free()


def test_kept_queues_of_a_search_are_idle_memory(hz, batch):
    batch.run("event", arena=(520 * MIB) // 64)
    before = free_mib()
    batch.run("event", arena=(520 * MIB) // 64)  # kept
    assert before == free_mib() < 600
    hz.Resident(pool_bytes=700 * MIB, arena_links=1 << 12).close()
    assert free_mib() > 900
    batch.run("event", arena=(520 * MIB) // 64)
    batch.run("event", arena=(400 * MIB) // 64)  # another size takes its place
    assert free_mib() < 700
    hz.check(hz.lib().hz_bfs_batch_release(batch.handle), "release")
    assert free_mib() > 900
