"""The norm bound that keeps states with infinite, NaN or huge amplitudes out
of the gate passes: its rule for written amplitudes on the CPU, and on the
device the gates after such a write."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

import qcs_amd
from qcs_amd import circuits as C

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_bound_rules(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "normbound_host")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra",
                    os.path.join(ROOT, "tests", "c", "normbound_host.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def real_gates():
    """H, RY and X have no imaginary part, so a NaN reaches the other part of
    an amplitude only as 0 * NaN."""
    ops = C.Ops()
    for q in (0, 1, 4):
        ops.add(C.H, q)
    ops.add(C.RY, 2, -1, 0.7)
    ops.add(C.X, 3)
    return ops


def gates_equal_one_by_one(prepare, ops=None, n=8):
    """``prepare`` sets both states up; the parts are compared each by itself
    (numpy calls two complex numbers with any NaN equal)."""
    ops = ops or real_gates()
    with qcs_amd.Circuit(n) as a, qcs_amd.Circuit(n) as b:
        prepare(a)
        prepare(b)
        a.apply(ops)
        for op, t, q, p in zip(ops.op, ops.tq, ops.cq, ops.par):
            b.apply(C.Ops().add(op, t, q, p))
            b.flush()
        x, y = a.amplitudes(), b.amplitudes()
    assert np.array_equal(x.real, y.real, equal_nan=True)
    assert np.array_equal(x.imag, y.imag, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [np.nan, np.inf, 1e300])
def test_finite_values_after_a_bad_one(qlib, bad):
    v = np.full(1 << 8, 0.0625, np.complex128)
    v[0] = bad  # (1e300: the NaN after it)
    v[1] = bad if bad != 1e300 else np.nan
    gates_equal_one_by_one(lambda c: c.set_amplitudes(v))


@pytest.mark.gpu
def test_part_of_a_nan_state_written(qlib):
    """A matrix with a NaN leaves half the state NaN; writing one amplitude
    does not make the rest finite.  Y and RZ have zeros in places where the
    per-gate kernels multiply NaN by them."""
    hip, _ = qlib
    m = (ctypes.c_double * 8)(1, 0, 0, 0, 0, 0, np.nan, 0)
    one = (ctypes.c_double * 2)(0.5, 0.25)

    def prepare(c):
        for q in range(c.n):
            c.h(q)
        assert hip.qcs_hip_apply_1q(c.device_state, c.n - 1, m) == 0
        assert hip.qcs_hip_write(c.device_state, 0, 1, one) == 0

    gates_equal_one_by_one(
        prepare, C.Ops().add(C.H, 0).add(C.Y, 7).add(C.RZ, 6, -1, 0.3).add(C.H, 3))
