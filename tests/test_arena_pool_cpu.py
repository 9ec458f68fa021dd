"""The arena that a context keeps between servers, and the library's device
allocations (csrc/arena_pool.hpp), on the CPU against a stand-in for the memory
calls, through tests/cpp/arena_pool_probe.  No GPU."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROBE = os.path.join(ROOT, "mcrg_amd", "_build", "arena_pool_probe")


@pytest.fixture(scope="module")
def lines():
    if not os.path.exists(PROBE):
        pytest.skip("mcrg_amd/_build/arena_pool_probe not built (make -C mcrg_amd)")
    out = subprocess.run([PROBE], capture_output=True, text=True, check=True, timeout=60).stdout
    return {line.split()[0]: line.split()[1:] for line in out.splitlines()}


def test_the_newest_arena_is_kept(lines):
    # bytes held and frees so far after servers of 40, 30, 30, 40 and 40 bytes
    assert lines["newest"] == ["40:0", "30:1", "30:1", "40:2", "40:2", "end", "0"]


def test_arenas_beyond_the_bound_are_freed(lines):
    # the small one stays while a larger one comes and goes; the largest kept replaces it
    assert lines["bounded"] == ["7", "1"]


def test_idle_arenas_go_when_memory_is_short(lines):
    # the first allocation of 90 bytes succeeds, the second cannot and reports it
    assert lines["pressure"] == ["0", "2", "1", "90", "50", "2"]


def test_tables_that_cannot_grow(lines):
    # 20 items, then 40 for 21; 60 cannot be had; then 10
    assert lines["table"] == ["0", "0", "40", "2", "0", "1", "0", "0", "10", "20"]


def test_every_allocation_may_use_the_idle_arena():
    src = os.path.join(ROOT, "mcrg_amd", "csrc")
    for name in os.listdir(src):
        if name != "arena_pool.hpp":
            with open(os.path.join(src, name)) as f:
                assert not re.search(r"\bhipMalloc\(", f.read()), name
