"""qcs_hip_measure_seq on qubits 0, 1, ... (joint weights, one collapse)
against qcs_hip_measure one after another: the same outcomes for the same
uniforms, and the same state to the rounding of the sums."""
import ctypes

import numpy as np
import pytest

import qcs_amd
from qcs_amd import circuits as C

pytestmark = pytest.mark.gpu


# sizes around the 10 bits a weight table covers, and one that needs the fold
@pytest.mark.parametrize("n,count", [(2, 2), (9, 9), (10, 10), (11, 11), (12, 3), (20, 20),
                                     (21, 13), (22, 22)])
def test_low_qubits_measured_together(qlib, n, count):
    hip, _ = qlib
    rng = np.random.default_rng(n * 100 + count)
    u = rng.random(count)
    u[0] = 1.0  # above every p0 < 1: outcome 1
    qs = (ctypes.c_int * count)(*range(count))
    got = (ctypes.c_int * count)()
    one = ctypes.c_int()
    with qcs_amd.Circuit(n) as a, qcs_amd.Circuit(n) as b:
        for c in (a, b):
            c.apply(C.layered(n, 2, n))
        assert hip.qcs_hip_measure_seq(a.device_state, count, qs,
                                       u.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), got) == 0
        for q in range(count):
            assert hip.qcs_hip_measure(b.device_state, q, u[q], ctypes.byref(one)) == 0
            assert one.value == got[q], q
        x, y = a.amplitudes(), b.amplitudes()
        assert np.max(np.abs(x - y)) <= 1e-13
        assert np.array_equal(x != 0, y != 0)


def test_basis_states_and_zero_weights(qlib):
    hip, _ = qlib
    n = 12
    u = np.full(n, 0.5)
    qs = (ctypes.c_int * n)(*range(n))
    got = (ctypes.c_int * n)()
    with qcs_amd.Circuit(n) as c:
        for basis in (0, 1, 0xA5C, (1 << n) - 1):
            c.set_basis_state(basis)
            assert hip.qcs_hip_measure_seq(c.device_state, n, qs,
                                           u.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                                           got) == 0
            assert list(got) == [(basis >> q) & 1 for q in range(n)]
            assert c.amplitudes()[basis] == 1.0 and c.norm_sq() == 1.0
