"""Batch records read one after the other (which brings the following jobs'
along) equal those read out of order, on both schedules, and follow the batch
when it runs on between the reads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _jobs(amd, n):
    # uneven sizes on the LDS-resident schedule, then shapes of the HBM schedule
    # whose blocks are short and long against their records
    jobs = [dict(L=(8, 16, 64, 8)[i % 4], coupling=0.44, seed=40 + i, n_therm=1, n_meas=3 + i % 5, n_levels=1 + i % 2,
                 sweeps_per_bin=2) for i in range(n)]
    jobs += [dict(L=L, coupling=0.43, seed=900 + 50 * L + i, n_therm=1, n_meas=6, n_levels=1, sweeps_per_bin=1,
                  sampler=amd.SAMPLER_SWENDSEN_WANG) for L in (4, 16, 256) for i in range(12)]
    return jobs


@pytest.mark.parametrize("n", [1, 2, 9, 700])
def test_sequential_reads_equal_single_reads(n):
    import mcrg_amd as amd
    print("read ahead", n, flush=True)
    with amd.Context(0) as ctx:
        jobs = _jobs(amd, n)
        with amd.Batch(ctx, jobs) as b:
            b.run(2)
            part = [b.records(i) for i in range(len(jobs))]
            b.run_all()
            full = [b.records(i) for i in range(len(jobs))]
            for i in reversed(range(len(jobs))):  # backwards: each read by itself
                assert np.array_equal(b.records(i), full[i]), i
            again = [b.records(i) for i in range(len(jobs))]
            assert all(np.array_equal(x, y) for x, y in zip(again, full))
            # samples counted in the last entry of each bin
            assert all(p[:, -1].sum() == min(1, j["n_meas"]) for p, j in zip(part, jobs))
            assert all(f[:, -1].sum() == j["n_meas"] for f, j in zip(full, jobs))
