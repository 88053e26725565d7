"""Job-table entries of the resident program reused while groups claim: some
hundreds of jobs of one start to 2^17 at once on one server, in both claim
orders, many more than the table's 64 entries. Every job ends, and its outputs
are its own."""

import numpy as np
import pytest

from test_resident_gpu import check_job

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("policy", ["RESIDENT_BY_ADMISSION", "RESIDENT_SMALLEST_FIRST"])
def test_entries_are_reused_under_claims(policy):
    import harmonize_amd as hz

    rng = np.random.default_rng(11)
    sizes = np.rint(2.0 ** rng.uniform(0.0, 17.0, size=400)).astype(int).tolist()
    res = hz.Resident(keep_outputs=True, policy=getattr(hz, policy))
    try:
        jobs = res.run_trace([(n, 3 + k) for k, n in enumerate(sizes)], np.zeros(len(sizes)), timeout_ms=10000.0)
        for k, (job, n) in enumerate(zip(jobs, sizes)):
            assert job["status"] == hz.JOB_DONE
            check_job(res, job["id"], n, 3 + k)
    finally:
        res.close()
