"""Several small lattices in one wave against the oracle: every number of them
that a launch takes (2 .. 64 of L = 8, 2 .. 16 of L = 16, 2 and 4 of L = 32),
with jobs that differ in thermalisation, length, bin size and coupling within
a wave, launches that stop anywhere, and a last wave that is partly empty."""
import math

import numpy as np
import pytest

KC = 0.5 * math.log(1.0 + math.sqrt(2.0))
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import mcrg_amd
    return mcrg_amd


def _group(L, n, waves):
    """Lattices a wave of n ones beside a larger lattice: as few as fit `waves` waves."""
    G = 4096 // L ** 2
    while G > 1 and -(-n // (G // 2)) <= waves:
        G //= 2
    return G


@pytest.mark.parametrize("L,G,nl,spl", [(8, 2, 2, 33), (8, 4, 2, 250), (8, 8, 1, 7), (8, 16, 2, 64), (8, 32, 0, 250),
                                        (8, 64, 2, 50), (16, 2, 3, 250), (16, 4, 2, 33), (16, 8, 3, 100),
                                        (16, 16, 3, 41), (32, 2, 4, 45), (32, 4, 3, 250)])
def test_groups_of_uneven_jobs(amd, orc, L, G, nl, spl):
    with amd.Context(0) as ctx:
        cus = ctx.device_info()["compute_units"]
        n = cus * G // 2 + G // 2 + max(1, G // 4)  # more than G / 2 a wave fit; the last wave partly empty
        assert _group(L, n, cus) == G and (G == 2 or n % G != 0)
        print("small groups", L, G, n, nl, spl, flush=True)
        jobs = [dict(L=L, coupling=(0.0, 0.3, KC, 0.7)[i % 4], seed=(i << 33) + 17 * i + L, n_therm=(0, 3, 70, 21)[i % 4],
                     n_meas=(1, 40, 90, 129)[(i // 3) % 4], n_levels=nl, sweeps_per_bin=(1, 5, 64, 1000)[(i // 2) % 4])
                for i in range(n)]
        jobs.append(dict(L=64, coupling=KC, seed=1, n_therm=5, n_meas=200, n_levels=2, sweeps_per_bin=100))
        # whole waves at the start, in the middle and at the end, and some of the rest
        look = sorted({i for a in (0, n // 2, n - 4 * G) for i in range(a, min(n, a + 4 * G))} |
                      set(range(0, n, max(1, n // 200))) | {n - 1, n})
        with amd.Batch(ctx, jobs, sweeps_per_launch=spl) as b:
            b.run_all()
            b.sync()
            for i in look:
                j = jobs[i]
                s_ref, r_ref = orc.run_chain(j["L"], j["coupling"], j["seed"], j["n_therm"], j["n_meas"], j["n_levels"],
                                             j["sweeps_per_bin"])
                assert np.array_equal(b.spins(i), s_ref), (i, j)
                assert np.array_equal(b.records(i), r_ref), (i, j)
