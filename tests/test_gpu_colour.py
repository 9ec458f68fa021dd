"""int8 chains of L = 64 and 128 in one workgroup, a set of waves per colour,
against the oracle: runs shorter and longer than the ring of buffers and the
blocks of samples, bins that several measuring waves share, every level count,
couplings with hardly any and with many undecided sites, and groups."""
import math

import numpy as np
import pytest

KC = 0.5 * math.log(1.0 + math.sqrt(2.0))
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import mcrg_amd
    return mcrg_amd


@pytest.fixture(scope="module")
def ctx(amd):
    with amd.Context(0) as c:
        yield c


@pytest.mark.parametrize("L", [64, 128])
@pytest.mark.parametrize("runs,spb,J,nl", [((1, 2, 3), 4, KC, 5), ((7, 1, 8, 9, 13), 50, KC, 0), ((300,), 7, 0.2, 1),
                                           ((255, 257), 1, 1.5, 2), ((600,), 1000, KC, 4), ((65,), 3, 0.0, 3),
                                           ((64, 70), 100, 0.004, 5)])
def test_chains(amd, ctx, orc, L, runs, spb, J, nl):
    print("colour chain", L, runs, spb, J, nl, flush=True)
    n = sum(runs)
    with amd.Chain(ctx, L, J, (7 << 40) + L, n_levels=nl, sweeps_per_bin=spb, max_bins=amd.n_bins(n, spb)) as ch:
        ch.sweep(1)
        ch.sweep(20)
        for r in runs:
            ch.sweep(r, measure=True)
        s_ref, r_ref = orc.run_chain(L, J, (7 << 40) + L, 21, n, nl, spb)
        assert ch.state() == (21 + n, n)
        assert np.array_equal(ch.spins(), s_ref)
        assert np.array_equal(ch.records(), r_ref)


@pytest.mark.parametrize("L,n_jobs", [(64, 3), (128, 5)])
def test_groups(amd, ctx, orc, monkeypatch, L, n_jobs):
    print("colour groups", L, n_jobs, flush=True)
    monkeypatch.setenv("MCRG_BATCH_RESIDENT", "0")
    jobs = [dict(L=L, coupling=(KC, 0.3, 0.7)[i % 3], seed=99 + i, n_therm=30, n_meas=90, n_levels=5, sweeps_per_bin=40)
            for i in range(n_jobs)]
    with amd.Batch(ctx, jobs, sweeps_per_launch=33) as b:
        b.run_all()
        b.sync()
        for i, j in enumerate(jobs):
            s_ref, r_ref = orc.run_chain(L, j["coupling"], j["seed"], 30, 90, 5, 40)
            assert np.array_equal(b.spins(i), s_ref), j
            assert np.array_equal(b.records(i), r_ref), j
