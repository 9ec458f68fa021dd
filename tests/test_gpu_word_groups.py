"""Words decided four at a time with their late ranks drawn together: strips
with four and more words a thread and one-wave lattices of L = 128, against
the oracle at couplings from hardly any open sites to nearly all."""
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


@pytest.mark.parametrize("J", [0.0, 0.004, 0.2, KC, 1.3])
@pytest.mark.parametrize("L,strips", [(512, 2), (1024, 2), (1024, 4), (1024, 8)])
def test_strips(amd, ctx, orc, monkeypatch, L, strips, J):
    print("word groups", L, strips, J, flush=True)
    monkeypatch.setenv("MCRG_STRIP_WG", str(strips))
    with amd.Chain(ctx, L, J, 9, n_levels=3, sweeps_per_bin=4, max_bins=1) as ch:
        ch.sweep(5)
        ch.sweep(3, measure=True)
        s_ref, r_ref = orc.run_chain(L, J, 9, 5, 3, 3, 4)
        assert np.array_equal(ch.spins(), s_ref)
        assert np.array_equal(ch.records(), r_ref)


@pytest.mark.parametrize("J", [0.0, 0.004, 0.2, KC, 1.3])
def test_waves(amd, ctx, orc, J):
    print("word groups: waves", J, flush=True)
    jobs = [dict(L=128, coupling=J, seed=41 * i, n_therm=20, n_meas=30, n_levels=6, sweeps_per_bin=10)
            for i in range(3)]
    with amd.Batch(ctx, jobs) as b:
        b.run_all()
        b.sync()
        for i, j in enumerate(jobs):
            s_ref, r_ref = orc.run_chain(128, J, j["seed"], 20, 30, 6, 10)
            assert np.array_equal(b.spins(i), s_ref)
            assert np.array_equal(b.records(i), r_ref)
