"""Gate-pass plans on the CPU: tests/c/gateplan_host.cpp plans random gate
lists with the planner of the gate passes, runs each pass's program the way
the kernel does (threads, registers, LDS slots, conditions, index maps) and
compares the state, value for value, with the gates applied one by one."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pass_programs_equal_gate_by_gate(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "gateplan_host")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-ffp-contract=off",
                    os.path.join(ROOT, "tests", "c", "gateplan_host.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("ok ")
