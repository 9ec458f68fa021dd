"""The work that users of mcrg_amd have it do, as cases that can be timed.

Every case runs through the package's public classes (Context, Chain, Batch,
Server).  Kinds:

  step    one sweep of one chain, then its operators: what the class interface
          does for each logged configuration (sample_new_configuration, then
          calc_energy), and what anyone does who looks at a chain sweep by sweep
  chain   one chain's next record bin: measured sweeps, then its records and
          spins (the checkpoint that is kept per bin)
  therm   thermalisation of a large chain: unmeasured sweeps, then the operators
          that say whether it has settled
  batch   a whole job list: the batch made, run to its end, every job's records
          read (what calc_critical_exponent's replicas are)
  serve   a burst of jobs through the job server: submitted, scheduled until
          all are done, their records fetched and released

Outputs are whole numbers (spins and int64 sums), equal for equal seeds, so no
value in 64-bit floating point stands beside them.
"""
import math

import numpy as np

import mcrg_amd as mc
from mcrg_amd.workloads import splitmix64, unit

KC = 0.5 * math.log(1.0 + math.sqrt(2.0))
# T/Tc = 1.02, 1.00, 0.98, 0.94, 0.90
COUPLINGS = (0.4320459, 0.4406868, 0.4496804, 0.4688157, 0.489652)
MASK = (1 << 64) - 1

_context = None


def _ctx():
    """One context for the process, as a user's program has."""
    global _context
    if _context is None:
        _context = mc.Context(0)
    return _context


def listed():
    return [
        # the 8 x 8 chain with one blocking: the smallest measured run
        dict(name="chain_8", kind="chain", L=8, levels=1, sweeps=1000, sampler=0, J=0.4406868),
        # one configuration at a time through the class interface
        dict(name="step_32", kind="step", L=32, J=KC),
        # the reference's N = 128 with all its levels, one chain, near K = -0.44
        dict(name="chain_128", kind="chain", L=128, levels=6, sweeps=500, sampler=0, J=0.44),
        # one cluster-sampled chain, as calc_critical_exponent runs it with one replica
        dict(name="chain_sw_64", kind="chain", L=64, levels=5, sweeps=200, sampler=1, J=KC),
        # the large single chain with five blockings
        dict(name="chain_2048", kind="chain", L=2048, levels=5, sweeps=1000, sampler=0, J=0.4406868),
        # the largest lattice, being thermalised
        dict(name="therm_16384", kind="therm", L=16384, sweeps=32, J=0.4406868),
        # 4096 replicas of uneven size and coupling, blocked down to L = 4
        dict(name="batch_mixed", kind="batch", jobs=4096, L_min=8, L_max=128, sampler=0, therm=1000, meas=10000,
             bin=1000),
        # many replicas of one small lattice (the exponent tables at N = 16)
        dict(name="batch_16", kind="batch", jobs=1024, L_min=16, L_max=16, sampler=0, therm=1000, meas=5000, bin=500),
        # lattices that fill a workgroup's share of LDS
        dict(name="batch_512", kind="batch", jobs=256, L_min=512, L_max=512, sampler=0, therm=100, meas=400, bin=100),
        # cluster-sampled replicas (the exponent tables at N = 16 .. 128)
        dict(name="batch_sw_64", kind="batch", jobs=1024, L_min=64, L_max=64, sampler=1, therm=20, meas=180, bin=60),
        # one round of the critical-coupling bisection: large lattices with the
        # cluster sampler beside small ones with Metropolis, matched levels
        dict(name="bisect_round", kind="bisect", large=64, small=1024, therm_large=10, meas_large=90, therm_small=500,
             meas_small=100),
        # requests of uneven size through the server
        dict(name="serve_burst", kind="serve", jobs=400, L_min=16, L_max=512, therm=100, meas_min=100, meas_max=2000,
             bin=50),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c):
    """About the microseconds of a pass: 800 site updates a nanosecond with
    Metropolis, 50 with the cluster sampler, and no sweep below a latency."""
    def us(sites, sweeps, sampler, lists=1):
        return max(sites * sweeps / (5e4 if sampler else 8e5), sweeps * lists * (40 if sampler else 15))

    if c["kind"] in ("step", "therm", "chain"):
        return us(c["L"] ** 2, c.get("sweeps", 1), c.get("sampler", 0))
    if c["kind"] == "bisect":
        return us(c["large"] * 1024 ** 2, c["therm_large"] + c["meas_large"], 1) + us(
            c["small"] * 128 ** 2, c["therm_small"] + c["meas_small"], 0)
    sites = c["jobs"] * _mean_sites(c["L_min"], c["L_max"])
    if c["kind"] == "batch":
        sizes = int(math.log2(c["L_max"] // c["L_min"])) + 1
        return 30 * c["jobs"] + us(sites, c["therm"] + c["meas"], c["sampler"], sizes if c["sampler"] else 1)
    return us(sites, c["therm"] + 0.5 * (c["meas_min"] + c["meas_max"]), 0)


def _mean_sites(lo, hi):
    k = range(int(math.log2(lo)), int(math.log2(hi)) + 1)
    return sum(4 ** i for i in k) / len(k)


def draw(rng):
    while True:
        kind = rng.choice(["chain", "chain", "batch", "batch", "batch", "step", "therm", "serve", "bisect"])
        J = round(rng.uniform(0.42, 0.47), 7)
        if kind == "step":
            c = dict(kind=kind, L=1 << rng.randint(3, 11), J=J)
        elif kind == "therm":
            L = 1 << rng.randint(10, 14)
            c = dict(kind=kind, L=L, sweeps=_log_int(rng, 3, max(4, min(2000, (1 << 34) // L ** 2))), J=J)
        elif kind == "chain":
            sampler = int(rng.random() < 0.3)
            k = rng.randint(3, 10 if sampler else 12)
            c = dict(kind=kind, L=1 << k, levels=rng.randint(1, k - 1), sweeps=_log_int(rng, 5, 800), sampler=sampler,
                     J=J)
        elif kind == "batch":
            sampler = int(rng.random() < 0.3)
            # Metropolis jobs up to L = 512, now and then of L = 1024
            top = 10 if sampler or rng.random() < 0.15 else 9
            a, b = sorted((rng.randint(3, top), rng.randint(3, top)))
            if b == 10:
                a = 10
            meas = _log_int(rng, 20, 5000)
            c = dict(kind=kind, jobs=_log_int(rng, 8, 4096 if b < 10 else 64), L_min=1 << a, L_max=1 << b,
                     sampler=sampler, therm=meas // 5, meas=meas, bin=max(1, meas // rng.randint(1, 12)))
        elif kind == "serve":
            a, b = sorted((rng.randint(4, 9), rng.randint(4, 9)))
            lo = _log_int(rng, 50, 500)
            c = dict(kind=kind, jobs=_log_int(rng, 10, 800), L_min=1 << a, L_max=1 << b, therm=_log_int(rng, 20, 200),
                     meas_min=lo, meas_max=lo * rng.randint(2, 20), bin=rng.randint(20, 100))
        else:
            c = dict(kind=kind, large=4 * rng.randint(1, 16), small=16 * rng.randint(4, 64),
                     therm_large=rng.randint(1, 10), meas_large=rng.randint(5, 60), therm_small=rng.randint(50, 400),
                     meas_small=rng.randint(20, 100))
        # at most the largest listed pass
        if _cost(c) <= 2e5 and c.get("meas_max", 0) <= 3000:
            return c


class _State:
    def __init__(self, case, seed):
        self.case, self.chain, self.jobs = case, None, None
        r = np.random.default_rng(seed)
        self.seed = int(r.integers(1, 1 << 62))
        k = case["kind"]
        if k in ("step", "therm", "chain"):
            L = case["L"]
            # bins long enough for any number of passes (int64-safe: shorter
            # ones, and more of them, on the largest lattices)
            bins = 4 if L <= 1024 else 64
            spb = min(1 << 28, mc.max_sweeps_per_bin(L))
            self.chain = mc.Chain(_ctx(), L, case["J"], self.seed, n_levels=case.get("levels", 0),
                                  sweeps_per_bin=spb, max_bins=bins if k == "chain" else 1,
                                  sampler=case.get("sampler", 0))
            self.chain.sweep(20)  # a chain in use is past its random start
            self.chain.sync()
        elif k in ("batch", "serve"):
            a, b = int(math.log2(case["L_min"])), int(math.log2(case["L_max"]))
            self.jobs = []
            for i in range(case["jobs"]):
                # the job list is the case's; the chains' random streams are the seed's
                h = splitmix64(i)
                L = 1 << (a + h % (b - a + 1))
                if k == "batch":
                    J, meas = COUPLINGS[(h >> 32) % 5], case["meas"]
                else:
                    J = 0.42 + 0.05 * unit(h)
                    meas = case["meas_min"] + splitmix64(h ^ 1) % (case["meas_max"] - case["meas_min"] + 1)
                self.jobs.append(dict(L=L, coupling=J, seed=(self.seed + i) & MASK, n_therm=case["therm"], n_meas=meas,
                                      n_levels=int(math.log2(L // 4)), sweeps_per_bin=case["bin"],
                                      sampler=case.get("sampler", 0)))
        else:
            # 16 couplings across the bracket, the lattices of each size shared
            # out among them; L = 1024 is blocked 3 + m times, L = 128 m times
            self.jobs = []
            for i in range(case["large"]):
                self.jobs.append(dict(L=1024, coupling=0.43 + 0.02 * (i % 16) / 15.0, seed=(self.seed + i) & MASK,
                                      n_therm=case["therm_large"], n_meas=case["meas_large"], n_levels=6,
                                      sweeps_per_bin=max(1, case["meas_large"] // 3), sampler=1))
            for i in range(case["small"]):
                self.jobs.append(dict(L=128, coupling=0.43 + 0.02 * (i % 16) / 15.0,
                                      seed=(self.seed + 100000 + i) & MASK, n_therm=case["therm_small"],
                                      n_meas=case["meas_small"], n_levels=3,
                                      sweeps_per_bin=max(1, case["meas_small"] // 4), sampler=0))

    def __del__(self):
        if self.chain is not None:
            self.chain.close()
            self.chain = None


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    c = state.case
    if c["kind"] == "step":
        state.chain.sweep(1)
        return state.chain.operators()
    if c["kind"] == "therm":
        state.chain.sweep(c["sweeps"])
        return state.chain.operators()
    if c["kind"] == "chain":
        state.chain.sweep(c["sweeps"], measure=True)
        return dict(records=state.chain.records(), spins=state.chain.spins())
    if c["kind"] == "serve":
        with mc.Server(_ctx()) as s:
            ids = [s.submit(j) for j in state.jobs]
            while s.step() > 0:
                pass
            out = []
            for i in ids:
                out.append(s.records(i).ravel())
                s.release(i)
        return np.concatenate(out)
    with mc.Batch(_ctx(), state.jobs) as b:
        b.run_all()
        return np.concatenate([b.records(i).ravel() for i in range(len(state.jobs))])


def work(case):
    """Bytes: the chains' spins read and written once (one byte a site where
    the chain holds int8, one bit otherwise) and the records out.  Operations:
    per 32 sites of a half-sweep one Philox call (10 rounds of 2 products, 2
    three-way exclusive-ors) and about 40 bit operations, i.e. 2.5 a site; a
    measured sweep adds about 30 per 32 sites."""
    k = case["kind"]

    def rec(levels):
        return 8 * (22 * levels + 16)

    def ops(sites, therm, meas):
        return sites * (2.5 * (therm + meas) + 1.0 * meas)

    if k in ("step", "therm"):
        n = case["L"] ** 2
        return dict(bytes=2 * n, flops=ops(n, case.get("sweeps", 1), 0))
    if k == "chain":
        n = case["L"] ** 2
        return dict(bytes=3 * n + rec(case["levels"]), flops=ops(n, 0, case["sweeps"]))
    if k == "bisect":
        b = case["large"] * (2 * 1024 ** 2 + 4 * rec(6)) + case["small"] * (128 ** 2 // 4 + 5 * rec(3))
        return dict(bytes=b, flops=case["large"] * ops(1024 ** 2, case["therm_large"], case["meas_large"]) +
                    case["small"] * ops(128 ** 2, case["therm_small"], case["meas_small"]))
    a, b = int(math.log2(case["L_min"])), int(math.log2(case["L_max"]))
    meas = case["meas"] if k == "batch" else 0.5 * (case["meas_min"] + case["meas_max"])
    n, bins = _mean_sites(case["L_min"], case["L_max"]), math.ceil(meas / case["bin"])
    levels = 0.5 * (a + b) - 2
    per = n * (2.0 if case.get("sampler") or n > 512 ** 2 else 0.25) + bins * rec(levels)
    return dict(bytes=case["jobs"] * per, flops=case["jobs"] * ops(n, case["therm"], meas))
