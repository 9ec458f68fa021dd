"""Servers that come after one another take over the job arena: fresh results
whatever the last one left there, also when its budget differs and when two
live at once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import mcrg_amd
    return mcrg_amd


def _job(L, seed):
    return dict(L=L, coupling=0.44, seed=seed, n_therm=3, n_meas=9, n_levels=2, sweeps_per_bin=4)


def _check(orc, srv, jobs):
    ids = [srv.submit(j) for j in jobs]
    while srv.step() > 0:
        pass
    for i, j in zip(ids, jobs):
        _, ref = orc.run_chain(j["L"], j["coupling"], j["seed"], 3, 9, 2, 4)
        assert np.array_equal(srv.records(i), ref), j
        srv.release(i)


@pytest.mark.parametrize("budgets", [(0, 0, 0), (1 << 26, 1 << 27, 1 << 26), (5 << 30, 5 << 30)])
def test_in_turn(amd, orc, budgets):
    print("arena pool", budgets, flush=True)
    with amd.Context(0) as ctx:
        for k, b in enumerate(budgets):
            with amd.Server(ctx, hbm_budget_bytes=b) as srv:
                _check(orc, srv, [_job(L, 7 * k + L) for L in (8, 64, 256)])


def test_at_once(amd, orc):
    print("arena pool: two servers", flush=True)
    with amd.Context(0) as ctx:
        with amd.Server(ctx) as a, amd.Server(ctx) as b:
            _check(orc, a, [_job(32, 1)])
            _check(orc, b, [_job(32, 2)])
        with amd.Server(ctx) as a, amd.Server(ctx) as b:
            _check(orc, a, [_job(128, 3)])
            _check(orc, b, [_job(128, 4)])
