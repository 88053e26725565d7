"""EventProgram's default number of groups is resident at once: a large
generation on it takes no longer than on an eighth fewer, which would not be so
if a few groups ran in a round of their own. Step counts are exact."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

COUNT = 1 << 24


def test_no_last_round_of_a_few_groups():
    import harmonize_amd as hz

    starts = hz.collatz_make_starts(21, 32, COUNT)
    steps = hz.DeviceArray(COUNT, np.uint32)
    cus = hz.device_facts()["compute_units"]

    def best_ms(groups):
        return min(hz.collatz_run("event", steps, starts, COUNT, groups=groups, max_launches=1 << 16)["elapsed_ms"]
                   for _ in range(3))

    fewer = best_ms(28 * cus)
    # Resident, 32 groups per CU hide more and take about as long; a round of
    # the last eighth of the groups takes a sixth longer.
    assert best_ms(32 * cus) < 1.08 * fewer
    want, _ = O.collatz_steps(O.collatz_make_starts(21, 32, 1 << 20))
    assert np.array_equal(steps.numpy()[:1 << 20], want)
