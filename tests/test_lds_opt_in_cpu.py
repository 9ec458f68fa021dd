"""Kernels with more than 64 KiB of dynamic LDS are opted in for it before their
launch, on every device (csrc/lds_opt_in.hpp, through
tests/cpp/lds_opt_in_probe).  No GPU."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROBE = os.path.join(ROOT, "mcrg_amd", "_build", "lds_opt_in_probe")


def test_levels_rise_on_each_device():
    if not os.path.exists(PROBE):
        pytest.skip("mcrg_amd/_build/lds_opt_in_probe not built (make -C mcrg_amd)")
    out = subprocess.run([PROBE], capture_output=True, text=True, check=True, timeout=60).stdout
    got = [tuple(map(int, line.split())) for line in out.splitlines()]
    assert got == [(0, 65536, 0, 0, 0),       # nothing to ask for
                   (0, 70000, 0, 70000, 1), (0, 66000, 0, 70000, 1),
                   (1, 66000, 0, 66000, 2),   # the other device has a level of its own
                   (1, 90000, 0, 90000, 3), (0, 80000, 0, 80000, 4), (1, 80000, 0, 90000, 4),
                   (0, 200000, 1, 80000, 5),  # refused: returned, and the level stays
                   (0, 80000, 0, 80000, 5), (0, 100000, 0, 100000, 6)]


@pytest.mark.parametrize("source,kernel", [("colour_kernels.hip", "k_colour_chain<L>"), ("resident_kernels.hip", "k_resident<NT>"),
                                           ("strip_kernels.hip", "k_strip<NT>"), ("sw_kernels.hip", "k_sw_wg<PW>")])
def test_launchers_ask(source, kernel):
    with open(os.path.join(ROOT, "mcrg_amd", "csrc", source)) as f:
        text = f.read()
    assert re.search(r"\.need\(reinterpret_cast<const void \*>\(&" + re.escape(kernel) + r"\), lds_bytes\)", text)
