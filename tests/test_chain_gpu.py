"""Lane chaining of the async program type: lanes run their successor promise
from registers and are filled again from the stash. Collatz starts whose chains
end together, one lane at a time, at once or never together, at counts around
a wavefront and a link, with cycle budgets that end launches between passes;
exact against the step counts and promise counts of the oracle."""

import numpy as np
import pytest

import harmonize_amd as hz
import oracle_lib as O

pytestmark = pytest.mark.gpu


def check(host, **cfg):
    ref, promises = O.collatz_steps(host)
    dev = hz.DeviceArray.from_numpy(host)
    steps = hz.DeviceArray(host.size, np.uint32)
    st = hz.collatz_run("async", steps, dev, flags=hz.RUN_AUDIT, max_launches=100000, **cfg)
    assert np.array_equal(steps.numpy(), ref)
    assert st["promises"] == promises
    assert st["audits"] == st["launches"]
    return st


@pytest.mark.parametrize("count", [1, 2, 63, 64, 65, 127, 4097])
@pytest.mark.parametrize("what", ["zero", "one", "same", "ramp", "overflow"])
def test_chain_ends(count, what):
    host = {
        "zero": np.zeros(count, np.uint64),                        # ends where it starts, an even value
        "one": np.ones(count, np.uint64),
        "same": np.full(count, 27, np.uint64),                     # every lane ends in the same pass
        "ramp": np.arange(count, dtype=np.uint64),                 # lanes end one by one
        "overflow": np.where(np.arange(count) % 3 == 0, np.uint64(12327829503), np.uint64(2**64 - 1)),
    }[what]
    check(host)


@pytest.mark.parametrize("cycles", [1, 2, 7])
def test_chain_survives_short_launches(cycles):
    # Lanes give their promises back when a launch ends, wherever it ends.
    host = O.collatz_make_starts(3, 40, 3001)
    st = check(host, cycles=cycles, groups=5, arena=4096)
    assert st["launches"] > 1 and st["spills"] == st["fills"] > 0


@pytest.mark.parametrize("coalesce", [1, 63, 64])
def test_chain_coalesce_thresholds(coalesce):
    check(O.collatz_make_starts(9, 32, 10007), coalesce=coalesce, groups=3)
