"""States that start as a basis state skip tiles of zeros until the gates have
mixed every qubit.  The same gates on the same state set through
qc_set_amplitudes (nothing known about it) give the same amplitudes, bit for
bit, whatever comes between them."""
import numpy as np
import pytest

import qcs_amd
from qcs_amd import circuits as C

pytestmark = pytest.mark.gpu

FORMS = [qcs_amd.PLAIN_FP64, qcs_amd.PLAIN_FP32, qcs_amd.FUSED_FP32,
         qcs_amd.FUSED_FP32 | qcs_amd.FUSE_TILES, qcs_amd.FUSED_FP32 | qcs_amd.FUSE_SPLIT_BF16]


def few_qubits(n, qubits, seed):
    """gates on some qubits only, controlled by others"""
    ops = C.Ops()
    rng = np.random.default_rng(seed)
    for q in qubits:
        ops.add(C.RY, q, -1, float(rng.uniform(-3, 3)))
        ops.add(C.P, (q + 3) % n, -1, float(rng.uniform(-3, 3)))
        ops.add(C.CNOT, q, (q + 5) % n)
        ops.add(C.CPHASE, (q + 7) % n, q, float(rng.uniform(-3, 3)))
        ops.add(C.H, q)
    ops.add(C.SWAP, qubits[0], (qubits[0] + 2) % n)
    ops.add(C.X, qubits[-1])
    return ops


@pytest.mark.parametrize("option", FORMS)
@pytest.mark.parametrize("n,basis", [(16, 0), (17, 0x1A5C3), (20, 0xFFFFF)])
def test_basis_state_equals_any_state(qlib, n, basis, option):
    v = np.zeros(1 << n, np.complex128)
    v[basis] = 1.0
    with qcs_amd.Circuit(n, option) as a, qcs_amd.Circuit(n, option) as b:
        a.set_basis_state(basis)
        b.set_amplitudes(v)
        for qubits in ([0], [n - 1, 3], [7, 8, 9], list(range(0, n, 3)), list(range(n))):
            ops = few_qubits(n, qubits, len(qubits))
            a.apply(ops)
            b.apply(ops)
            assert np.array_equal(a.amplitudes(), b.amplitudes()), qubits
        # a new basis state after a full one
        a.set_basis_state(1)
        ops = few_qubits(n, [2, n - 2], 9)
        a.apply(ops)
        v[basis] = 0.0
        v[1] = 1.0
        b.set_amplitudes(v)
        b.apply(ops)
        assert np.array_equal(a.amplitudes(), b.amplitudes())


@pytest.mark.parametrize("option", [qcs_amd.PLAIN_FP64, qcs_amd.FUSED_FP32 | qcs_amd.FUSE_TILES])
def test_calls_that_fill_the_state(qlib, option):
    """After Grover rounds, written amplitudes, a dense unitary or a matrix
    with an infinite entry every tile counts again."""
    hip, _ = qlib
    n = 16
    ops = few_qubits(n, [4, 9], 2)
    u = np.eye(2) * (1 / np.sqrt(2))
    u[0, 1], u[1, 0] = 1 / np.sqrt(2), -1 / np.sqrt(2)
    m = np.ascontiguousarray(u.astype(np.complex128)).view(np.float64)

    def grover(c):
        assert hip.qcs_hip_grover(c.device_state, 5, 1) == 0

    def write(c):
        c.set_amplitudes(np.array([0.5, 0.25j]), 40000)

    def unitary(c):
        q = np.array([15], np.int32)
        import ctypes
        assert hip.qcs_hip_apply_unitary(c.device_state, 1,
                                         q.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
                                         m.ctypes.data_as(ctypes.POINTER(ctypes.c_double))) == 0

    for between in (grover, write, unitary):
        with qcs_amd.Circuit(n, option) as a, qcs_amd.Circuit(n, option) as b:
            v = np.zeros(1 << n, np.complex128)
            v[3] = 1.0
            a.set_basis_state(3)
            b.set_amplitudes(v)
            for c in (a, b):
                c.apply(ops)
                between(c)
                c.apply(ops)
            assert np.array_equal(a.amplitudes(), b.amplitudes()), between.__name__
            assert abs(a.norm_sq() - b.norm_sq()) == 0.0


@pytest.mark.parametrize("option,n", [(qcs_amd.PLAIN_FP64, 21), (qcs_amd.PLAIN_FP32, 22),
                                      (qcs_amd.FUSED_FP32 | qcs_amd.FUSE_TILES, 22)])
def test_zeros_that_no_pass_wrote(qlib, option, n):
    """A large basis state starts without its zeros in memory (here full of
    another state's amplitudes): every call sees them all the same."""
    hip, _ = qlib
    basis = 0x155A5A & ((1 << n) - 1)
    v = np.zeros(1 << n, np.complex128)
    v[basis] = 1.0
    full = C.Ops()
    for q in range(n):
        full.add(C.H, q)

    def near(c, ops):
        c.apply(ops)
        return c.amplitudes()

    some = few_qubits(n, [1, 2, 9, 17], 3)
    swap = C.Ops().add(C.SWAP, 0, n - 1)
    calls = {
        "read": lambda c: c.amplitudes(),
        "part": lambda c: c.amplitudes((1 << n) - 5000, 5000),
        "norm": lambda c: np.array([c.norm_sq()]),
        "probability": lambda c: np.array([c.get_probability_l(basis), c.get_probability_l(3)]),
        "most likely": lambda c: np.array([c.find_most_likely_state_l()]),
        "sample": lambda c: c.sample_indices(16),
        "one pass": lambda c: near(c, some),
        "one gate": lambda c: near(c, C.Ops().add(C.H, n - 1)),
        "swap": lambda c: near(c, swap),
        "all qubits": lambda c: near(c, full),
        "measure": lambda c: np.concatenate([c.measure_all_list(), c.amplitudes().view(float)]),
        "pass, measure": lambda c: (c.apply(some), c.measure_all_list(), c.amplitudes())[2],
        "write": lambda c: (c.set_amplitudes(np.ones(3, complex), 77), c.amplitudes())[1],
        "grover": lambda c: np.array([hip.qcs_hip_grover(c.device_state, 5, 2), *c.amplitudes(0, 9)]),
        "overflow": lambda c: (huge(hip, c), c.amplitudes())[1],
    }
    with qcs_amd.Circuit(n, option) as a, qcs_amd.Circuit(n, option) as b:
        for name, call in calls.items():
            for c in (a, b):
                c.apply(full)
                c.lib.qc_flush(c.handle)
            a.set_basis_state(basis)
            b.set_amplitudes(v)
            libc = qcs_amd.libc()
            libc.srand(7)
            x = call(a)
            libc.srand(7)
            y = call(b)
            assert np.array_equal(x, y, equal_nan=True), name


def huge(hip, c):
    import ctypes
    m = (ctypes.c_double * 8)(1e200, 0, 0, 0, 0, 0, 1e200, 0)
    if c.options & 1 == 0:  # (a matrix beyond the bound of queued gates)
        for _ in range(2):
            assert hip.qcs_hip_apply_1q(c.device_state, 1, m) == 0
