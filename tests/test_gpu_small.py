"""Small lattices in the registers of a wave (L = 8, 16, 32) against the
oracle: every number of lattices per wave and lanes per lattice, bins shorter
than a block of samples and ending inside it, jobs of one wave that differ in
phase and length, launches that stop anywhere, and the int8 chains."""
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


@pytest.mark.parametrize("L", [8, 16, 32])
@pytest.mark.parametrize("n_jobs,max_group,spl", [(1, 0, 250), (3, 64, 7), (5, 2, 100), (64, 0, 33), (300, 0, 64),
                                                  (700, 1, 250)])
def test_batches(amd, ctx, orc, L, n_jobs, max_group, spl):
    print("small batch", L, n_jobs, max_group, spl, flush=True)
    top = int(math.log2(L)) - 1
    jobs = [dict(L=L, coupling=(0.0, 0.3, KC, 0.7)[i % 4], seed=(i << 33) + 17 * i + L, n_therm=(0, 3, 70)[i % 3],
                 n_meas=(1, 40, 90, 129)[(i // 3) % 4], n_levels=top - i % 2 * (top > 1) if n_jobs < 100 else top,
                 sweeps_per_bin=(1, 5, 64, 1000)[(i // 2) % 4]) for i in range(n_jobs)]
    with amd.Batch(ctx, jobs, sweeps_per_launch=spl, max_group=max_group) as b:
        b.run_all()
        b.sync()
        for i in range(n_jobs) if n_jobs < 70 else list(range(0, n_jobs, 37)) + [n_jobs - 1]:
            j = jobs[i]
            s_ref, r_ref = orc.run_chain(L, j["coupling"], j["seed"], j["n_therm"], j["n_meas"], j["n_levels"],
                                         j["sweeps_per_bin"])
            assert np.array_equal(b.spins(i), s_ref), j
            assert np.array_equal(b.records(i), r_ref), j


@pytest.mark.parametrize("L", [8, 16, 32])
@pytest.mark.parametrize("runs,spb,J", [((1, 2, 3), 4, KC), ((63, 1, 64, 65), 50, KC), ((130,), 7, 0.2), ((70, 70), 1, 1.5)])
def test_chains(amd, ctx, orc, L, runs, spb, J):
    print("small chain", L, runs, spb, J, flush=True)
    for nl in (0, 1, int(math.log2(L)) - 1):
        n = sum(runs)
        with amd.Chain(ctx, L, J, 5 + L, n_levels=nl, sweeps_per_bin=spb, max_bins=amd.n_bins(n, spb)) as ch:
            ch.sweep(1)
            ch.sweep(67)
            for r in runs:
                ch.sweep(r, measure=True)
            s_ref, r_ref = orc.run_chain(L, J, 5 + L, 68, n, nl, spb)
            assert ch.state() == (68 + n, n)
            assert np.array_equal(ch.spins(), s_ref)
            assert np.array_equal(ch.records(), r_ref)
