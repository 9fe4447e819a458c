"""The queue of plain gates on the CPU: tests/c/gatequeue_host.cpp pushes gates
and takes passes as the backend does; the queue keeps to its limit."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_queue_keeps_to_its_limit(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "gatequeue_host")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra",
                    os.path.join(ROOT, "tests", "c", "gatequeue_host.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
