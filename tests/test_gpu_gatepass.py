"""Gate passes (many plain gates per sweep over the state) against the gates
applied one by one: a flush after every gate leaves one gate in the queue,
which runs in its per-gate kernel.  The amplitudes are equal, value for value
(the arithmetic is the same; only a zero's sign may differ)."""
import ctypes

import numpy as np
import pytest

import qcs_amd
from oracle.oracle import OracleState
from qcs_amd import circuits as C

pytestmark = pytest.mark.gpu

KINDS = [C.H, C.X, C.Y, C.Z, C.P, C.RX, C.RY, C.RZ, C.CNOT, C.CPHASE, C.SWAP]


def one_by_one(c, ops):
    for op, t, q, p in zip(ops.op, ops.tq, ops.cq, ops.par):
        one = C.Ops().add(op, t, q, p)
        c.apply(one)
        c.flush()


# 7: the smallest queued state (8 threads); 10: one full wave; 13, 14: the
# largest single tile and the first state of two; 17: tiles in a wider state.
# 1500 gates overrun the queue's limit.
@pytest.mark.parametrize("n,count", [(7, 300), (8, 200), (10, 300), (12, 1500), (13, 300),
                                     (14, 300), (17, 400)])
def test_random_circuits_equal_the_oracle(qlib, n, count):
    ops = C.random_circuit(n, count, 100 + n, KINDS)
    st = OracleState(n)
    st.run(ops)
    with qcs_amd.Circuit(n) as c:
        c.apply(ops)
        assert np.array_equal(c.amplitudes(), st.vector())


@pytest.mark.parametrize("option", [qcs_amd.PLAIN_FP64, qcs_amd.PLAIN_FP32])
@pytest.mark.parametrize("n", [9, 13, 16, 21])
def test_passes_equal_per_gate_kernels(qlib, n, option):
    parts = [C.random_circuit(n, 120, 7 * n, KINDS), C.layered(n, 2, n), C.qft(n, swaps=True)]
    with qcs_amd.Circuit(n, option) as a, qcs_amd.Circuit(n, option) as b:
        for ops in parts:
            a.apply(ops)
            one_by_one(b, ops)
            assert np.array_equal(a.amplitudes(), b.amplitudes())


@pytest.mark.parametrize("n", [24, 27])
def test_large_states_with_index_maps(qlib, n):
    """CNOTs folded into a pass's stores, many work-groups at once: a store
    may hit what another wave of the work-group still has to load."""
    ops = C.layered(n, 1, 3)
    for q in range(n - 1):
        ops.add(C.CNOT, (q + 7) % n, q)
    with qcs_amd.Circuit(n) as a, qcs_amd.Circuit(n) as b:
        a.apply(ops)
        one_by_one(b, ops)
        omf, mx = a.compare_with(b)
        assert mx == 0.0 and abs(a.norm_sq() - 1.0) < 1e-12


def test_every_way_of_looking_sees_the_queued_gates(qlib):
    hip, _ = qlib
    n = 11
    x = (ctypes.c_double * 8)(0, 0, 1, 0, 1, 0, 0, 0)
    with qcs_amd.Circuit(n) as c:
        st = c.device_state
        for k, look in enumerate([lambda: c.get_probability(want) == 1.0,
                                  lambda: c.find_most_likely_state() == want,
                                  lambda: list(c.sample_indices(3)) == [want] * 3,
                                  lambda: c.amplitudes()[want] == 1.0,
                                  lambda: c.measure(0) == want % 2,
                                  lambda: c.measure_all_list() ==
                                  [(want >> q) & 1 for q in range(n)]]):
            want = 1 + k
            c.set_basis_state(0)
            for q in range(n):
                if (want >> q) & 1:
                    assert hip.qcs_hip_apply_1q(st, q, x) == 0
            assert look(), k


def test_values_that_could_overflow_take_the_per_gate_kernels(qlib):
    """Infinite and NaN amplitudes, and matrices that grow the state, spread
    as the per-gate arithmetic spreads them (0 times infinity is NaN)."""
    n = 8
    rng = np.random.default_rng(2)
    for bad in (np.inf, np.nan, 1e300):
        v = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
        v[5] = bad
        with qcs_amd.Circuit(n) as a, qcs_amd.Circuit(n) as b:
            a.set_amplitudes(v)
            b.set_amplitudes(v)
            ops = C.layered(n, 2, 1)
            a.apply(ops)
            one_by_one(b, ops)
            assert np.array_equal(a.amplitudes(), b.amplitudes(), equal_nan=True)
    hip, _ = qlib
    big = (ctypes.c_double * 8)(1e200, 0, 0, 0, 0, 0, 1e200, 0)
    with qcs_amd.Circuit(n) as a, qcs_amd.Circuit(n) as b:
        for c, each in ((a, False), (b, True)):
            st = c.device_state
            for q in range(4):
                c.h(q)
                assert hip.qcs_hip_apply_1q(st, q, big) == 0
                if each:
                    c.flush()
        assert np.array_equal(a.amplitudes(), b.amplitudes(), equal_nan=True)


@pytest.mark.parametrize("option", [qcs_amd.PLAIN_FP64, qcs_amd.PLAIN_FP32])
@pytest.mark.parametrize("n", [14, 15, 18, 23])
def test_swaps_of_qubits_outside_the_tile(qlib, n, option):
    """Passes that store their tiles in each other's place: from a basis state
    and from any state, against the gates launched one by one."""
    rng = np.random.default_rng(n)
    start = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    start /= np.linalg.norm(start)
    for rep in range(6):
        ops = C.Ops()
        for _ in range(40):
            k, t = rng.integers(0, 8), int(rng.integers(0, n))
            c = int((t + rng.integers(1, n)) % n)
            if k < 5:
                ops.add(C.SWAP, t, c)
            elif k == 5:
                ops.add(C.H, t)
            elif k == 6:
                ops.add(C.CNOT, t, c)
            else:
                ops.add(C.CPHASE, t, c, float(rng.uniform(-3, 3)))
        if rep == 0:  # a bit reversal
            ops = C.Ops()
            for q in range(n // 2):
                ops.add(C.SWAP, q, n - 1 - q)
        with qcs_amd.Circuit(n, option) as a, qcs_amd.Circuit(n, option) as b:
            for c in (a, b):
                if rep < 4:
                    c.set_amplitudes(start)
                else:
                    c.set_basis_state(rep * 1234 % (1 << n))
            a.apply(ops)
            for op, t, c, p in zip(ops.op, ops.tq, ops.cq, ops.par):
                b.apply(C.Ops().add(op, t, c, p))
                b.lib.qc_flush(b.handle)
            assert np.array_equal(a.amplitudes(), b.amplitudes()), rep
