"""Which schedule a batch's jobs take follows MCRG_BATCH_RESIDENT at the batch's
creation, whatever earlier batches of the process took, and groups of one-wave
and one-workgroup int8 lattices equal the oracle."""
import math

import numpy as np
import pytest

KC = 0.5 * math.log(1.0 + math.sqrt(2.0))
pytestmark = pytest.mark.gpu
HALF_SWEEP, RESIDENT = 0, 3  # kernel kinds of mcrg_ctx_kernel_time


@pytest.fixture(scope="module")
def amd():
    import mcrg_amd
    return mcrg_amd


@pytest.mark.parametrize("L,n_jobs", [(8, 5), (16, 3), (32, 70), (64, 3), (128, 5)])
def test_schedule_of_each_batch(amd, orc, monkeypatch, L, n_jobs):
    top = int(math.log2(L)) - 1
    jobs = [dict(L=L, coupling=(KC, 0.3, 0.7)[i % 3], seed=99 + i, n_therm=30, n_meas=90, n_levels=top, sweeps_per_bin=40)
            for i in range(n_jobs)]
    ref = {}
    for i in sorted({0, 1, n_jobs // 2, n_jobs - 1}):
        ref[i] = orc.run_chain(L, jobs[i]["coupling"], jobs[i]["seed"], 30, 90, top, 40)
    for value in (None, "0", "1", "0"):
        print("schedule", L, n_jobs, value, flush=True)
        if value is None:
            monkeypatch.delenv("MCRG_BATCH_RESIDENT", raising=False)
        else:
            monkeypatch.setenv("MCRG_BATCH_RESIDENT", value)
        with amd.Context(0) as ctx:
            ctx.set_timing(True)
            with amd.Batch(ctx, jobs, sweeps_per_launch=33) as b:
                b.run_all()
                b.sync()
                for i, (s, r) in ref.items():
                    assert np.array_equal(b.spins(i), s), (value, i)
                    assert np.array_equal(b.records(i), r), (value, i)
            on = [ctx.kernel_time(k)[0] > 0 for k in (HALF_SWEEP, RESIDENT)]
            assert on == ([True, False] if value == "0" else [False, True]), value
