"""The resident program's list of jobs, whose places the housekeeping pass reads,
tests and moves together: jobs of one start to many that end in any order,
more of them than the list has places, in both claim orders. Every job's
outputs are exact."""

import pytest

from test_resident_gpu import check_job

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("policy", ["RESIDENT_BY_ADMISSION", "RESIDENT_SMALLEST_FIRST"])
@pytest.mark.parametrize("sizes", [[1] * 70, [65, 1, 4097, 64, 63] * 13, [1 << 19, 3, 1 << 17, 20000] * 16])
def test_jobs_come_and_go(policy, sizes):
    import harmonize_amd as hz

    res = hz.Resident(keep_outputs=True, policy=getattr(hz, policy))
    try:
        ids = [res.submit(n, 7 + k) for k, n in enumerate(sizes)]
        res.drain(60000)
        for k, (job, n) in enumerate(zip(ids, sizes)):
            check_job(res, job, n, 7 + k)
    finally:
        res.close()
