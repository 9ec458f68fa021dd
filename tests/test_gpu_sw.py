"""Swendsen-Wang kernels against the oracle's sequential union-find, at the
sizes where they can go wrong: lattices smaller than a word or a wave, the
first and last size of each kernel, single domains and no bonds at all, bins
that end inside and between launches, and every workgroup size of a batch."""
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


def _chain(amd, ctx, orc, L, J, seed, therm, runs, nl, spb):
    n = sum(runs)
    with amd.Chain(ctx, L, J, seed, n_levels=nl, sweeps_per_bin=spb, max_bins=amd.n_bins(n, spb),
                   sampler=amd.SAMPLER_SWENDSEN_WANG) as ch:
        ch.sweep(therm)
        for r in runs:
            ch.sweep(r, measure=True)
        s, rec = ch.spins(), ch.records()
        assert ch.state() == (therm + n, n)
    s_ref, r_ref = orc.run_chain(L, J, seed, therm, n, nl, spb, sampler=orc.SAMPLER_SW)
    assert np.array_equal(s, s_ref)
    assert np.array_equal(rec, r_ref)


@pytest.mark.parametrize("L", [2, 4, 8, 16, 32, 64, 128])
@pytest.mark.parametrize("J", [0.0, KC, 3.0])
def test_small_lattices(amd, ctx, orc, L, J):
    nl = max(0, int(math.log2(L)) - 1)
    print("sw", L, J, flush=True)
    _chain(amd, ctx, orc, L, J, 901 + L, 3, (5, 1, 9), nl, 4)


@pytest.mark.parametrize("L,n_jobs", [(8, 40), (16, 700), (64, 300), (64, 1500), (128, 600)])
def test_batches_of_every_workgroup_size(amd, ctx, orc, L, n_jobs):
    print("sw batch", L, n_jobs, flush=True)
    jobs = [dict(L=L, coupling=0.40 + 0.001 * (i % 80), seed=5000 + i, n_therm=2, n_meas=5, n_levels=2,
                 sweeps_per_bin=3, sampler=amd.SAMPLER_SWENDSEN_WANG) for i in range(n_jobs)]
    with amd.Batch(ctx, jobs, sweeps_per_launch=3) as b:
        b.run_all()
        b.sync()
        for i in sorted({0, 1, n_jobs // 2, n_jobs - 1}):
            j = jobs[i]
            s_ref, r_ref = orc.run_chain(L, j["coupling"], j["seed"], 2, 5, 2, 3, sampler=orc.SAMPLER_SW)
            assert np.array_equal(b.spins(i), s_ref), i
            assert np.array_equal(b.records(i), r_ref), i


@pytest.mark.parametrize("L,J,runs", [(256, 0.0, (2, 3)), (256, KC, (1, 40)), (256, 3.0, (3, 1)), (256, 0.35, (2, 2)),
                                      (512, KC, (4, 1)), (512, 0.6, (2,)), (1024, 0.47, (2,))])
def test_tiled_lattices(amd, ctx, orc, L, J, runs):
    """Lattices of 64 x 64 tiles: no bonds, one domain, clusters of every size;
    runs shorter and longer than a captured graph, which hand the spins over
    as int8."""
    print("sw tiles", L, J, runs, flush=True)
    _chain(amd, ctx, orc, L, J, 77 + L, 2, runs, 3, 4)


@pytest.mark.parametrize("L,n_jobs", [(256, 33), (512, 9)])
def test_tiled_batches(amd, ctx, orc, L, n_jobs):
    """Enough tiles for the launch shape of many lattices."""
    print("sw tiled batch", L, n_jobs, flush=True)
    jobs = [dict(L=L, coupling=0.43 + 0.001 * i, seed=31 + i, n_therm=1, n_meas=3, n_levels=4, sweeps_per_bin=2,
                 sampler=amd.SAMPLER_SWENDSEN_WANG) for i in range(n_jobs)]
    with amd.Batch(ctx, jobs, sweeps_per_launch=2) as b:
        b.run_all()
        b.sync()
        for i in (0, n_jobs // 2, n_jobs - 1):
            j = jobs[i]
            s_ref, r_ref = orc.run_chain(L, j["coupling"], j["seed"], 1, 3, 4, 2, sampler=orc.SAMPLER_SW)
            assert np.array_equal(b.spins(i), s_ref), i
            assert np.array_equal(b.records(i), r_ref), i
