"""Lattices of L = 256 and 512 in a workgroup's LDS against the oracle: every
workgroup size and level count, bins that end inside a block of 64 samples,
launches that stop anywhere, slots in parts."""
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


@pytest.mark.parametrize("L", [256, 512])
@pytest.mark.parametrize("threads,spl,parts", [(64, 250, 0), (128, 33, 0), (256, 250, 4), (512, 70, 0), (1024, 250, 0),
                                               (1024, 21, 3)])
def test_large_slots(amd, ctx, orc, L, threads, spl, parts):
    print("large slots", L, threads, spl, parts, flush=True)
    top = int(math.log2(L)) - 1
    jobs = [dict(L=L, coupling=(KC, 0.3, 0.0)[i % 3], seed=(i << 33) + 17 * i + L, n_therm=(0, 3, 20)[i % 3],
                 n_meas=(1, 66, 129)[(i // 2) % 3], n_levels=nl, sweeps_per_bin=(5, 100, 1)[(i // 3) % 3])
            for i, nl in enumerate([0, 1, 2, 3, 4, 5, top - 1, top, top, top])]
    with amd.Batch(ctx, jobs, threads=min(threads, 512), threads_large=threads, sweeps_per_launch=spl,
                   sub_chunks=parts) as b:
        b.run_all()
        b.sync()
        for i, j in enumerate(jobs):
            s_ref, r_ref = orc.run_chain(L, j["coupling"], j["seed"], j["n_therm"], j["n_meas"], j["n_levels"],
                                         j["sweeps_per_bin"])
            assert np.array_equal(b.spins(i), s_ref), j
            assert np.array_equal(b.records(i), r_ref), j
