"""Gate passes at the sizes where the tile changes, against the per-gate
kernels and the oracle: value for value, as the arithmetic is the same."""
import numpy as np
import pytest

import qcs_amd
from oracle.oracle import OracleState
from qcs_amd import circuits as C

pytestmark = pytest.mark.gpu

KINDS = [C.H, C.X, C.Y, C.Z, C.P, C.RX, C.RY, C.RZ, C.CNOT, C.CPHASE, C.SWAP]


# One tile up to 12 qubits: 4 amplitudes a thread while 512 threads hold it
# (11: all nine thread bits), 16 at 12.  10-bit tiles with 4 a thread from 13
# (the first state of several tiles) to 19, 12-bit tiles with 16 from 20 on.
@pytest.mark.parametrize("option", [qcs_amd.PLAIN_FP64, qcs_amd.PLAIN_FP32])
@pytest.mark.parametrize("n", [7, 10, 11, 12, 13, 19, 20])
def test_passes_equal_per_gate_kernels(qlib, n, option):
    parts = [C.random_circuit(n, 200, 11 * n, KINDS), C.layered(n, 2, n), C.qft(n, swaps=True)]
    with qcs_amd.Circuit(n, option) as a, qcs_amd.Circuit(n, option) as b:
        for ops in parts:
            a.apply(ops)
            for op, t, q, p in zip(ops.op, ops.tq, ops.cq, ops.par):
                b.apply(C.Ops().add(op, t, q, p))
                b.flush()
            assert np.array_equal(a.amplitudes(), b.amplitudes())


@pytest.mark.parametrize("n", [11, 12, 13, 19, 20])
def test_random_circuits_equal_the_oracle(qlib, n):
    ops = C.random_circuit(n, 300, 500 + n, KINDS)
    st = OracleState(n)
    st.run(ops)
    with qcs_amd.Circuit(n) as c:
        c.apply(ops)
        assert np.array_equal(c.amplitudes(), st.vector())
