# SPDX-License-Identifier: Apache-2.0
"""The scratch pool's rules (csrc/kda_scratch.hip) on a model of the HIP runtime, on the CPU
(scratch_host.cpp): a block is never lent or freed before its last use, no call waits for another
stream's block or works on the null stream, a refused wait, free or record loses and reuses
nothing, the last release gives everything back, a call under capture keeps its own, and an
allocation that fails is tried again without the pool's idle blocks."""
from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "kimi-k3-in-c_amd" / "csrc"
CASES = ["reuse", "evict_leaves_blocks_in_flight", "evict_idle_blocks_on_the_calls_stream",
         "evict_own_block_in_flight", "refused_wait", "refused_free", "refused_record", "last_release", "capture",
         "out_of_memory", "out_of_memory_under_capture"]


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    exe = tmp_path_factory.mktemp("scratch") / "scratch_host"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wno-unused-result", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{CSRC}", "-x", "c++", str(HERE / "scratch_host.cpp"),
                    str(CSRC / "kda_scratch.hip"), "-o", str(exe)], check=True)
    assert subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split() == CASES
    return exe


@pytest.mark.parametrize("case", CASES)
def test_scratch_rules(host, case):
    r = subprocess.run([host, case], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0, r.stdout
