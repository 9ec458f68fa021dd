"""Rules by which launches are shaped, on the CPU through
tests/cpp/launch_rules_probe.  No GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROBE = os.path.join(ROOT, "mcrg_amd", "_build", "launch_rules_probe")
CU_LDS, UNIT = 160 * 1024, 1280


def _ask(lines):
    if not os.path.exists(PROBE):
        pytest.skip("mcrg_amd/_build/launch_rules_probe not built (make -C mcrg_amd)")
    out = subprocess.run([PROBE], input="".join(f"{x}\n" for x in lines), capture_output=True, text=True, check=True)
    return [int(x) for x in out.stdout.split()]


@pytest.mark.parametrize("cus", [256, 304, 64])
def test_cluster_workgroups_spread_and_leave_room(cus):
    cases = [(share, n, need) for share in range(1, 11) for n in (cus * (share - 1) + 1, cus * share)
             for need in (600, 9000, 40000, 130000)]
    for (share, n, need), got in zip(cases, _ask(f"sw_lds {need} {n} {cus}" for share, n, need in cases)):
        assert got >= need
        if share > 8:
            assert got == need
            continue
        taken = -(-got // UNIT) * UNIT
        # one more than an even share does not fit a compute unit, ...
        assert (share + 1) * taken > CU_LDS, (share, n, need, got)
        if got > need:
            # ... an even share does, and nothing is asked for beyond that:
            # about half of the unit is left beside one, a ninth beside eight
            assert share * taken <= CU_LDS
            assert CU_LDS - share * taken >= CU_LDS // (share + 1) - (share + 1) * UNIT, (share, got)
