"""Strip launches of every length, from one sweep on, and of every size, also
where a chain's sweeps take another route by themselves (MCRG_STRIP=1 asks for
strips): spins, counters and record bins against the oracle, and the launches
counted, so that no other route stands in."""
import math

import numpy as np
import pytest

KC = 0.5 * math.log(1.0 + math.sqrt(2.0))
pytestmark = pytest.mark.gpu
STRIP = 4  # kernel kind of mcrg_ctx_kernel_time


@pytest.fixture(scope="module")
def amd():
    import mcrg_amd
    return mcrg_amd


def _check(amd, orc, L, J, nl, seed, spb, runs):
    with amd.Context(0) as ctx:
        ctx.set_timing(True)
        n_meas, n = sum(k for k, m in runs if m), sum(k for k, _ in runs)
        s = orc.init_spins(L, seed)
        # the oracle's chain: unmeasured and measured runs in their order
        ref = np.zeros((amd.n_bins(n_meas, spb), amd.record_size(nl)), dtype=np.int64)
        t = q = 0
        with amd.Chain(ctx, L, J, seed=seed, n_levels=nl, sweeps_per_bin=spb, max_bins=ref.shape[0]) as ch:
            for k, measure in runs:
                for _ in range(k):
                    s, one = orc.run_chain(L, J, seed, 0 if measure else 1, 1 if measure else 0, nl, 1, s=s, t0=t)
                    if measure:
                        ref[q // spb] += one[0]
                        q += 1
                    t += 1
                ch.sweep(k, measure=measure)
                assert np.array_equal(ch.spins(), s), (k, measure)
                assert np.array_equal(ch.records(), ref), (k, measure)
            assert ch.state() == (n, n_meas)
        assert ctx.kernel_time(STRIP)[0] == len(runs)


@pytest.mark.parametrize("halo,split", [("1", "1"), ("1", "0"), ("0", "1")])
@pytest.mark.parametrize("L,nl", [(64, 0), (64, 5), (128, 3), (256, 4), (512, 5), (1024, 3), (2048, 5)])
def test_short_runs(amd, orc, monkeypatch, L, nl, halo, split):
    print("strip runs", L, nl, halo, split, flush=True)
    monkeypatch.setenv("MCRG_STRIP", "1")
    monkeypatch.setenv("MCRG_STRIP_HALO", halo)
    monkeypatch.setenv("MCRG_STRIP_SPLIT", split)
    _check(amd, orc, L, KC, nl, 77 + L, 4,
           [(1, True), (2, True), (1, False), (3, False), (3, True), (5, True), (13, True), (9, True)])


@pytest.mark.parametrize("J", [0.0, 0.004, 0.2, KC, 1.3])
@pytest.mark.parametrize("L,strips", [(512, 2), (1024, 2), (1024, 8), (4096, 256)])
def test_many_words_a_thread(amd, orc, monkeypatch, L, strips, J):
    print("strip words", L, strips, J, flush=True)
    monkeypatch.setenv("MCRG_STRIP", "1")
    monkeypatch.setenv("MCRG_STRIP_WG", str(strips))
    _check(amd, orc, L, J, 3, 9, 4, [(2, False), (3, True), (1, True)])


@pytest.mark.parametrize("L,nl", [(64, 5), (128, 0), (128, 6)])
def test_static_sweeps_of_small_lattices(amd, orc, L, nl):
    print("strip static", L, nl, flush=True)
    s_ref, r_ref = orc.run_chain(L, KC, 5 + L, 7, 12, nl, 5)
    with amd.Context(0) as ctx, amd.Chain(ctx, L, KC, seed=5 + L, n_levels=nl, sweeps_per_bin=5, max_bins=3) as ch:
        for k in (3, 4):
            ch.sweep_static(k)
        for k in (1, 2, 9):
            ch.sweep_static(k, measure=True)
        assert np.array_equal(ch.spins(), s_ref)
        assert np.array_equal(ch.records(), r_ref)
