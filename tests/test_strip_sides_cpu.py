"""Launch shapes with two measuring workgroups a strip and eight tails
(mcrg::strip_shape with sides = 2) on the CPU, through
tests/cpp/strip_shape_probe: the workspace holds every index that both
measuring workgroups of a strip use, and the slots keep the race bounds.  No
GPU."""
import math
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROBE = os.path.join(ROOT, "mcrg_amd", "_build", "strip_shape_probe")


@pytest.fixture(scope="module")
def shapes():
    if not os.path.exists(PROBE):
        pytest.skip("mcrg_amd/_build/strip_shape_probe not built (make -C mcrg_amd)")
    lines = [f"{1 << lg} {nl} {min(256, (1 << lg) // 2)} {tails} 1 1 1 {sides}\n" for lg in range(6, 14)
             for nl in range(0, lg - 1) for tails in (8, 4) for sides in (1, 2)]
    out = subprocess.run([PROBE], input="".join(lines), capture_output=True, text=True, check=True).stdout
    rows = [({k: int(v) for k, v in (f.split("=") for f in line.split()[1:])}) for line in out.splitlines()]
    assert len(rows) == 1 + len(lines)
    return rows[0], [(s, int(line.split()[7])) for s, line in zip(rows[1:], lines)]


def test_both_sides_fit_the_workspace(shapes):
    c, sh = shapes
    seen = set()
    for s, sides in sh:
        if not s["split"]:
            continue
        seen.add((s["L"], sides))
        assert s["split"] == sides and s["n_meas"] == sides * s["n_wg"]
        # one count a measuring workgroup, copies a strip, (data, seq) words
        assert s["o_snap"] - s["o_snapc"] >= s["n_meas"] * c["kStripFlagStride"]
        assert s["o_snap"] % 2 == 0
        assert s["ws_words"] - s["o_snap"] >= 2 * c["kStripSnapSlots"] * s["n_wg"] * s["snap_words"]
    # every size whose strips take measuring workgroups at all
    assert seen == {(1 << lg, k) for lg in range(6, 12) for k in (1, 2)}


def test_first_row_slots_outlast_both_sides(shapes):
    c, sh = shapes
    for s, sides in sh:
        if s["split"]:
            # the first rows of sample k are read before sample k + sides is
            # released; the lower strip may be kStripSnapSlots + 1 samples
            # further by then
            assert s["first_slots"] > sides + c["kStripSnapSlots"] + 1, s


def test_tails_share_the_ring(shapes):
    c, sh = shapes
    for s, _ in sh:
        # a slot belongs to one tail, so that its samples are taken in order
        assert c["kStripRing"] % s["n_tail"] == 0
        assert s["lam"] == min(int(math.log2(s["R"])), s["nl"])
