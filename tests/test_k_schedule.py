"""The K loop of the persistent grouped GEMM kernel takes its loads, reads, waits and barriers from csrc/k_schedule.hpp.
k_schedule_check.cpp walks the same functions on the host, for every number of K steps up to 12 and two tiles in a row: no
access to an operand tile may be ordered by time only."""

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "accelerated-model-architectures_amd", "csrc")


def _check(tmp_path, *defines):
    exe = str(tmp_path / "k_schedule_check")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, *defines, os.path.join(HERE, "k_schedule_check.cpp"), "-o", exe], check=True)
    return subprocess.run([exe], capture_output=True, text=True)


def test_every_access_is_ordered_by_a_barrier(tmp_path):
    r = _check(tmp_path)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("fault,says", [("-DPLANT_NO_BARRIER", "overwritten while another wave"), ("-DPLANT_IN_FLIGHT", "before the loads")])
def test_the_walk_finds_a_planted_fault(tmp_path, fault, says):
    r = _check(tmp_path, fault)
    assert r.returncode == 1 and says in r.stdout
