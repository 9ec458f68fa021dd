"""A chain's operators on demand against the spins they belong to, at every side
and row count a thread works off; chains beyond the context's result lines; and
runs of a few sweeps between long ones."""
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


def _operators(s):
    s = s.astype(np.int64)
    right, down = np.roll(s, -1, 1), np.roll(s, -1, 0)
    diag = np.roll(down, -1, 1)
    return [int((s * right).sum() + (s * down).sum()), int((s * diag).sum() + (right * down).sum()),
            int((s * right * down * diag).sum()), int(s.sum())]


@pytest.mark.parametrize("L", [2, 4, 8, 16, 32, 64, 128, 256, 512, 1024, 2048, 4096, 8192])
def test_operators(amd, ctx, L):
    print("operators", L, flush=True)
    with amd.Chain(ctx, L, 0.3, 11 + L, n_levels=min(1, int(math.log2(L)) - 1), sweeps_per_bin=1,
                   max_bins=1) as ch:
        for step in range(3):
            spins = ch.spins().reshape(L, L)
            assert [int(v) for v in ch.operators()] == _operators(spins), step
            assert [int(v) for v in ch.operators()] == _operators(spins), step
            ch.sweep(1, measure=step == 1)


def test_more_chains_than_lines(amd, ctx):
    print("operators: 70 chains", flush=True)
    chains = [amd.Chain(ctx, 16, 0.3, i) for i in range(70)]
    try:
        for c in chains:
            assert [int(v) for v in c.operators()] == _operators(c.spins().reshape(16, 16))
    finally:
        for c in chains:
            c.close()


@pytest.mark.parametrize("L", [256, 1024])
def test_short_runs(amd, ctx, orc, L):
    print("short runs", L, flush=True)
    runs = ((1, False), (5, False), (6, False), (1, True), (9, True), (2, True), (3, True), (2, True))
    with amd.Chain(ctx, L, KC, 3, n_levels=4, sweeps_per_bin=4, max_bins=5) as ch:
        for n, measure in runs:
            ch.sweep(n, measure=measure)
        s_ref, r_ref = orc.run_chain(L, KC, 3, 12, 17, 4, 4)
        assert np.array_equal(ch.spins(), s_ref)
        assert np.array_equal(ch.records(), r_ref)
