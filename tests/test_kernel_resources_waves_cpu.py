"""Register and scratch budgets of the kernels that hold lattices in waves and
workgroups, from hipcc's resource report for gfx950 (no GPU needed).

The budgets are what the kernels take.  k_wave (the batched workload) has four
waves on a SIMD and spills 23 registers at that, k_colour_chain<128> one.  More
would cost either of them.
"""
import re

import pytest

from test_kernel_resources_cpu import resources

# source, kernel, instances, VGPRs, scratch bytes a lane, waves per SIMD
BUDGETS = [
    ("wave_kernels.hip", r"6k_waveE", 1, 128, 60, 4),
    ("small_kernels.hip", r"k_small_chainILj8E", 1, 96, 0, 5),
    ("small_kernels.hip", r"k_small_chainILj(16|32)E", 2, 128, 0, 4),
    ("colour_kernels.hip", r"k_colour_chainILj64E", 1, 146, 0, 3),
    ("colour_kernels.hip", r"k_colour_chainILj128E", 1, 128, 8, 4),
    ("sw_kernels.hip", r"k_sw_wgI", 4, 82, 0, 5),
    ("sw_kernels.hip", r"k_sw_tileI", 2, 48, 0, 7),
    ("sw_kernels.hip", r"k_sw_(seam|apply|measure0)E", 3, 27, 0, 8),
]


@pytest.fixture(scope="module")
def report(tmp_path_factory):
    seen = {}

    def get(source):
        if source not in seen:
            seen[source] = resources(source, tmp_path_factory.mktemp("resources"))
        return seen[source]

    return get


@pytest.mark.parametrize("source,kernel,count,vgprs,scratch,waves", BUDGETS)
def test_budget(report, source, kernel, count, vgprs, scratch, waves):
    ks = {n: r for n, r in report(source).items() if re.search(kernel, n)}
    assert len(ks) == count, sorted(report(source))
    for name, r in ks.items():
        assert r["VGPRs"] <= vgprs and r["ScratchSize"] <= scratch and r["Occupancy"] >= waves, (name, r)
