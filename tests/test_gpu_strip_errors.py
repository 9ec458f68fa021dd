"""A strip launch whose waits give up (MCRG_STRIP_WAIT_TICKS=0 lets every wait
that is not over at once) leaves the chain's state lost: whatever reads the
chain next reports it, once, and other chains are not concerned."""
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


@pytest.mark.parametrize("reader", ["operators", "sync", "spins", "records"])
@pytest.mark.parametrize("lines", [True, False])
def test_lost_state_is_reported(amd, ctx, orc, monkeypatch, reader, lines):
    print("strip error", reader, lines, flush=True)
    L, J, seed = 1024, 0.44, 3
    # 64 chains of a context have a pinned line for their results
    others = [] if lines else [amd.Chain(ctx, 8, J, seed=i) for i in range(64)]
    try:
        with amd.Chain(ctx, L, J, seed=seed, n_levels=3, sweeps_per_bin=1000) as ch:
            monkeypatch.setenv("MCRG_STRIP_WAIT_TICKS", "0")
            ch.sweep(400, measure=True)
            with pytest.raises(amd.MCRGError) as e:
                getattr(ch, reader)()
            assert e.value.status == amd.ERR_DEVICE and "exceeded the limit" in str(e.value)
            ch.sync()
        monkeypatch.delenv("MCRG_STRIP_WAIT_TICKS")
        with amd.Chain(ctx, L, J, seed=seed, n_levels=3, sweeps_per_bin=1000) as ch:
            ch.sweep(9, measure=True)
            s_ref, r_ref = orc.run_chain(L, J, seed, 0, 9, 3, 1000)
            S = orc.ops(L, s_ref)
            assert tuple(ch.operators()[:3]) == tuple(S)
            assert np.array_equal(ch.spins(), s_ref)
            assert np.array_equal(ch.records(), r_ref)
    finally:
        for c in others:
            c.close()


@pytest.mark.parametrize("then", ["same", "larger"])
def test_a_later_launch_does_not_hide_it(amd, ctx, monkeypatch, then):
    """An error that nobody has asked about yet outlives the next launch, in the
    same workspace or in a larger one."""
    print("strip error, then", then, flush=True)
    with amd.Chain(ctx, 1024, 0.44, seed=3, n_levels=3, sweeps_per_bin=1000) as ch:
        monkeypatch.setenv("MCRG_STRIP_WAIT_TICKS", "0")
        if then == "larger":
            monkeypatch.setenv("MCRG_STRIP_WG", "8")
        ch.sweep(400, measure=True)
        monkeypatch.delenv("MCRG_STRIP_WAIT_TICKS")
        monkeypatch.delenv("MCRG_STRIP_WG", raising=False)
        with pytest.raises(amd.MCRGError) as e:
            ch.sweep(50, measure=True)
            ch.sync()
        assert e.value.status == amd.ERR_DEVICE
