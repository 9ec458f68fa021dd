"""One-workgroup chains of L = 64 and 128 whose waves give up on their waits for
each other (MCRG_COLOUR_SPINS=0 lets every wait that is not over at once): the
launch ends, the lattice stays as it was, and whatever reads it next reports
that, once."""
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


@pytest.mark.parametrize("L", [64, 128])
@pytest.mark.parametrize("reader,lines", [("operators", True), ("sync", True), ("spins", True), ("records", True),
                                          ("operators", False), ("records", False)])
def test_chain(amd, ctx, orc, monkeypatch, L, reader, lines):
    print("colour error", L, reader, lines, flush=True)
    J, seed = 0.44, 3
    # 64 chains of a context have a pinned line for their results and error word
    others = [] if lines else [amd.Chain(ctx, 8, J, seed=i) for i in range(64)]
    try:
        with amd.Chain(ctx, L, J, seed=seed, n_levels=3, sweeps_per_bin=1000) as ch:
            monkeypatch.setenv("MCRG_COLOUR_SPINS", "0")
            ch.sweep(50, measure=True)
            with pytest.raises(amd.MCRGError) as e:
                getattr(ch, reader)()
            assert e.value.status == amd.ERR_DEVICE and "exceeded the limit" in str(e.value)
            monkeypatch.delenv("MCRG_COLOUR_SPINS")
            ch.sync()
            assert np.array_equal(ch.spins(), orc.init_spins(L, seed))
            # the chain can be set up again and goes on
            ch.set_state(0, 0, np.zeros_like(ch.records()))
            ch.sweep(9, measure=True)
            s_ref, r_ref = orc.run_chain(L, J, seed, 0, 9, 3, 1000)
            assert np.array_equal(ch.spins(), s_ref)
            assert np.array_equal(ch.records(), r_ref)
    finally:
        for c in others:
            c.close()


@pytest.mark.parametrize("reader", ["spins", "records"])
def test_groups(amd, ctx, monkeypatch, reader):
    print("colour error: groups", reader, flush=True)
    monkeypatch.setenv("MCRG_BATCH_RESIDENT", "0")
    jobs = [dict(L=64, coupling=0.44, seed=i, n_therm=5, n_meas=20, n_levels=2, sweeps_per_bin=10) for i in range(3)]
    with amd.Batch(ctx, jobs) as b:
        monkeypatch.setenv("MCRG_COLOUR_SPINS", "0")
        b.run_all()
        with pytest.raises(amd.MCRGError) as e:
            getattr(b, reader)(1)
        assert e.value.status == amd.ERR_DEVICE
        getattr(b, reader)(2)
