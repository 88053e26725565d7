"""How EventProgram deals a generation to its groups: inputs around a link of
64 and around the 64 segments, fewer and more groups than links, several links
in a row, and generations launched a few at a time with a limit on launches.
Step counts are exact."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 63, 64, 65, 4095, 4097, 64 * 64 * 3 + 17])
@pytest.mark.parametrize("groups,cycles", [(1, 1), (3, 2), (64, 1), (1000, 3), (0, 0)])
def test_generation_parts(count, groups, cycles):
    import harmonize_amd as hz

    starts = np.random.default_rng(count).integers(1, 1 << 20, size=count, dtype=np.uint64)
    dev, steps = hz.DeviceArray.from_numpy(starts), hz.DeviceArray(count, np.uint32)
    st = hz.collatz_run("event", steps, dev, groups=groups, cycles=cycles, max_launches=1 << 16)
    want, promises = O.collatz_steps(starts)
    assert np.array_equal(steps.numpy(), want) and st["promises"] == promises
