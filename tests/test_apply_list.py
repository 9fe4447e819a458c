"""Circuit.apply hands a gate list to one C call (qc_apply_gates): the gates it
records, its messages and the exceptions are those of the qc_* calls made one
by one, whatever the lists hold.  (Deferred circuits: no device needed.)"""
import numpy as np
import pytest

import qcs_amd
from qcs_amd import circuits as C


class Lists:
    def __init__(self, op, tq, cq, par):
        self.op, self.tq, self.cq, self.par = op, tq, cq, par


def one_by_one(c, ops):
    for op, t, k, p in zip(ops.op, ops.tq, ops.cq, ops.par):
        c._dispatch[op](int(t), int(k), float(p))


def outcome(fn, make, capfd):
    capfd.readouterr()
    raised = None
    with qcs_amd.Circuit(5, qcs_amd.DEFERRED) as c:
        try:
            fn(c, make())
        except Exception as e:
            raised = type(e)
        c.lib.qc_print_circuit(c.handle)
        gates = c.lib.qc_get_num_gates(c.handle)
    qcs_amd.libc().fflush(None)
    out = capfd.readouterr()
    return raised, gates, out.out, out.err


def mixed():
    ops = C.Ops()
    for op in range(11):
        ops.add(op, op % 5, (op + 2) % 5, 0.25 * op)
    return ops


LISTS = {
    "every gate": mixed,
    "empty": lambda: C.Ops(),
    "invalid qubits": lambda: Lists([0, 8, 8, 10, 1], [5, 1, 9, 2, -1], [-1, 1, 0, 2, -1], [0.0] * 5),
    "unknown code": lambda: Lists([0, 11, 1], [0, 1, 2], [-1] * 3, [0.0] * 3),
    "negative code": lambda: Lists([0, -1, 1], [0, 1, 2], [-1] * 3, [0.0] * 3),
    "shortest list": lambda: Lists([0, 1, 2], [0, 1], [-1] * 5, [0.0] * 3),
    "arrays": lambda: Lists(*mixed().arrays()),
    "float qubits": lambda: Lists([0, 8.0], [1.7, 2.2], [-1.0, 3.9], [0, 1]),
    "wide qubit": lambda: Lists([0, 1], [1, 2**32 + 3], [-1, -1], [0.0, 0.0]),
    "bytes": lambda: Lists(bytes([0, 1, 4]), bytes([2, 3, 4]), [-1] * 3, bytes(3)),
    "generators": lambda: Lists(iter([0, 4]), iter([1, 2]), iter([-1, -1]), iter([0.0, 0.5])),
    "no angle": lambda: Lists([0, 5, 1], [1, 2, 3], [-1] * 3, [0.0, None, 0.0]),
    "text": lambda: Lists([0, 1], ["1", "2"], [-1, -1], ["0.5", "x"]),
    "no finite angle": lambda: Lists([4, 5], [1, 2], [-1] * 2, [np.inf, np.nan]),
}


@pytest.mark.parametrize("name", LISTS)
def test_list_equals_calls(name, capfd):
    a = outcome(lambda c, ops: c.apply(ops), LISTS[name], capfd)
    b = outcome(one_by_one, LISTS[name], capfd)
    assert a == b


def test_counts_the_gates_applied():
    _, q = qcs_amd.load()
    with qcs_amd.Circuit(3, qcs_amd.DEFERRED) as c:
        op, t, k = (np.array(x, np.int32) for x in ([0, 1, 99, 2], [0, 1, 2, 0], [-1] * 4))
        p = np.zeros(4)
        args = [x.ctypes.data for x in (op, t, k, p)]
        assert q.qc_apply_gates(c.handle, *args, 4) == 2
        assert q.qc_apply_gates(c.handle, *args, 0) == 0
        assert q.qc_get_num_gates(c.handle) == 2
        assert q.qc_apply_gates(None, *args, 1) == 1
        assert q.qc_apply_gates(c.handle, None, *args[1:], 1) == 0
