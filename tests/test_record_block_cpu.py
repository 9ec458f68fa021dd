"""Reading a batch's records ahead (mcrg::RecordBlock, csrc/record_block.hpp) on
the CPU, through tests/cpp/record_block_probe: what a read gives is what the
device holds at that moment, also when reads come while a run is in progress,
and a block that cannot be had is replaced by single reads.  No GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROBE = os.path.join(ROOT, "mcrg_amd", "_build", "record_block_probe")


@pytest.fixture(scope="module")
def lines():
    if not os.path.exists(PROBE):
        pytest.skip("mcrg_amd/_build/record_block_probe not built (make -C mcrg_amd)")
    out = subprocess.run([PROBE], capture_output=True, text=True, check=True, timeout=60).stdout
    return {line.split()[0]: line.split()[1:] for line in out.splitlines()}


def test_sequence_comes_in_blocks(lines):
    got = dict(f.split("=") for f in lines["sequence"])
    assert got["same"] == "1"
    # windows of 1, 8, 64, 512, 4096 jobs
    assert (int(got["singles"]), int(got["blocks"])) == (1, 4)


def test_reads_during_a_run_are_not_kept(lines):
    # during the run 1 then 2, whatever was read before; behind it 3
    assert lines["progress"] == ["1"] * 4 + ["2"] * 3 + ["3"] * 6


def test_overlapping_runs(lines):
    assert lines["overlap"] == ["2", "2", "2"]


def test_runs_drop_blocks(lines):
    assert lines["between"] == ["9", "9"]


def test_without_a_block(lines):
    # no memory, no contiguous range, a failed copy (its error is returned)
    assert lines["memory"] == ["4"] * 5 + ["-107"] + ["4"] * 2
