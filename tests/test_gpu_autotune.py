"""The autotuner tries only configurations whose launches differ, and the options
that have no effect on launches are still checked and reported."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import mcrg_amd
    return mcrg_amd


@pytest.fixture(scope="module")
def ctx(amd):
    with amd.Context(0) as c:
        yield c


# what is tried: the configuration in use twice, then 128, 256 and 512 threads for
# L = 256 and for L = 512 (1024 in use while there are few), and 256 with 512
@pytest.mark.parametrize("Ls,threads,tries", [((8, 32, 128), 0, 2), ((64,), 512, 2), ((256, 8), 0, 4), ((512,), 0, 5),
                                              ((256, 512), 0, 6)])
def test_only_different_launches_are_tried(amd, ctx, orc, Ls, threads, tries):
    print("autotune", Ls, threads, flush=True)
    jobs = [dict(L=L, coupling=0.44, seed=7 * i + L, n_therm=3, n_meas=17, n_levels=2, sweeps_per_bin=10)
            for i in range(2) for L in Ls]
    with amd.Batch(ctx, jobs, threads=threads, sweeps_per_launch=2, autotune=True) as b:
        n = 0
        while b.options()["autotune"]:
            b.run(2)
            n += 1
        assert n == tries
        b.run_all()
        b.sync()
        opts = b.options()
        if max(Ls) <= 128:
            assert (opts["threads"], opts["threads_large"]) == (threads or 256, 0)
        # what it reports is accepted
        amd.Batch(ctx, jobs[:1], **{k: opts[k] for k in ("threads", "max_slot_lds", "min_team", "max_team", "threads_large",
                                                        "sub_chunks")}).close()
        for i, j in enumerate(jobs):
            s_ref, r_ref = orc.run_chain(j["L"], 0.44, j["seed"], 3, 17, 2, 10)
            assert np.array_equal(b.spins(i), s_ref)
            assert np.array_equal(b.records(i), r_ref)


def test_options_without_effect(amd, ctx):
    jobs = [dict(L=16, coupling=0.44, seed=1, n_therm=0, n_meas=4, n_levels=1, sweeps_per_bin=4)]
    with amd.Batch(ctx, jobs, threads=128, min_team=32, max_team=64, max_slot_lds=4096) as b:
        o = b.options()
        assert (o["min_team"], o["max_team"], o["max_slot_lds"]) == (32, 64, 4096)
    for bad in (dict(min_team=3), dict(min_team=512), dict(max_team=8), dict(max_slot_lds=-1)):
        with pytest.raises(amd.MCRGError) as e:
            amd.Batch(ctx, jobs, **bad)
        assert e.value.status == amd.ERR_INVALID_ARG
