"""The barrier program where ids are claimed for several steps at once: counts
around a wavefront and a claim, more barriers than dependents, one barrier for
all (whose semaphore a wavefront updates at once), and launches that end with
claimed ids not started. Every held promise runs once, after its release."""

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dep,non,barriers", [(0, 1, 1), (1, 0, 3), (63, 65, 64), (511, 2, 1), (4097, 0, 1),
                                              (0, 70001, 5), (40003, 20021, 7)])
@pytest.mark.parametrize("cfg", [{}, {"groups": 5, "cycles": 3}, {"groups": 333, "queues": 3}])
def test_counts(dep, non, barriers, cfg):
    import harmonize_amd as hz

    if dep + non > 40000 and "cycles" in cfg:
        # Steps started in place are not queued promises, and a run of which
        # two launches evaluate none of those is refused.
        with pytest.raises(hz.HarmonizeError, match="no progress"):
            hz.barrier_run(dep, non, barriers, max_launches=1 << 16, flags=hz.RUN_AUDIT, **cfg)
        return
    counter, hits, violations, st = hz.barrier_run(dep, non, barriers, max_launches=1 << 16, flags=hz.RUN_AUDIT, **cfg)
    assert counter == 2 * dep + non and violations == 0
    assert (hits == 1).all() and st["audits"] == st["launches"]
