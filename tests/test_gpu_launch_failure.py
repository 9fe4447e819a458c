"""States after a launch that reports a failure: what is known of their zeros,
and the calls that replace them.

The failure is injected on the host (QCS_HIP_INJECT_FAULT=launch:N: the N-th
launch check of the process fails although the kernel ran), so the amplitudes
may or may not have spread: the passes that follow must not leave tiles out
as zeros.  Each case runs in a child process; the device never faults."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# H on the qubits of the first launch, which reports the failure, then H on
# the others: the uniform state if the launch ran and is not taken for lost
CHILD = r"""
import sys
sys.path.insert(0, %r)
import numpy as np
import qcs_amd
n, option, first, rest = 14, %d, %s, %s
c = qcs_amd.Circuit(n, option)
q, h = c.lib, c.handle
for t in first:
    q.qc_h(h, t)
q.qc_flush(h)
print("ERR", q.qc_last_error(h), flush=True)
for t in rest:
    q.qc_h(h, t)
q.qc_flush(h)
a = c.amplitudes()
print("OFF", float(np.max(np.abs(a - 2.0 ** (-n / 2)))), flush=True)
"""


@pytest.mark.parametrize("option,launch,tol", [(0x0, 2, 1e-15), (0x1, 3, 1e-8)])
def test_a_failed_launch_leaves_no_tile_out(qlib, option, launch, tol):
    # launch checks: 1 = |0> fill of qc_create; complex128: 2 = the pass of the
    # first gates, on one tile of 10 bits; fused complex64: 2 = the composition,
    # 3 = the block of the first five
    first = list(range(10)) if option == 0 else list(range(5, 10))
    rest = [10, 11, 12, 13] + [q for q in range(5) if q not in first]
    code = CHILD % (ROOT, option, first, rest)
    env = dict(os.environ, QCS_HIP_INJECT_FAULT=f"launch:{launch}")
    p = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True,
                       timeout=120)
    assert p.returncode == 0, p.stderr
    assert "ERR -4" in p.stdout and p.stderr.count("injected failure") == 1, p.stdout + p.stderr
    assert float(p.stdout.split("OFF ")[1].split()[0]) <= tol


REPLACE = r"""
import sys
sys.path.insert(0, %r)
import ctypes
import numpy as np
import qcs_amd
n, how = 8, %r
c = qcs_amd.Circuit(n)
q, h = c.lib, c.handle
for t in range(n):
    q.qc_h(h, t)
want = np.zeros(1 << n, np.complex128)
want[5] = 1.0
if how == "basis":
    c.set_basis_state(5)
else:
    q.qc_set_amplitudes(h, 0, 1 << n, want.ctypes.data_as(ctypes.POINTER(ctypes.c_double)))
print("ERR", q.qc_last_error(h), flush=True)
a = c.amplitudes()
c.h(0)
c.h(0)
print("SAME", bool(np.array_equal(a, want)), abs(c.amplitudes()[5] - 1.0) < 1e-15, flush=True)
"""


@pytest.mark.parametrize("how", ["basis", "write"])
def test_a_replaced_state_does_not_need_the_gates_before(qlib, how):
    """The queued gates' failure (launch check 2) is reported by the call that
    launches them, a reset or a write of the whole state, which still does
    what it was called for."""
    env = dict(os.environ, QCS_HIP_INJECT_FAULT="launch:2")
    p = subprocess.run([sys.executable, "-c", REPLACE % (ROOT, how)], env=env,
                       capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr
    assert "ERR -4" in p.stdout and p.stderr.count("injected failure") == 1, p.stdout + p.stderr
    assert "SAME True True" in p.stdout, p.stdout


SYNC = r"""
import sys
sys.path.insert(0, %r)
import time
import qcs_amd
hip, q = qcs_amd.load()
a, b = qcs_amd.Circuit(8), qcs_amd.Circuit(28)
b.flush()
for t in range(8):
    a.h(t)
for t in range(28):
    b.h(t)
    b.ry(t, 0.3)
t0 = time.perf_counter()
rc = hip.qcs_hip_device_sync()
t1 = time.perf_counter()
b.flush()
t2 = time.perf_counter()
print("RC", rc, "FIRST", t1 - t0 > t2 - t1, flush=True)
"""


def test_device_sync_waits_for_every_state(qlib):
    """Launch check 3 is the pass of the first state; the second one's passes
    (4 GiB, milliseconds) are launched and waited for all the same, so the
    flush after it finds nothing to do."""
    env = dict(os.environ, QCS_HIP_INJECT_FAULT="launch:3")
    p = subprocess.run([sys.executable, "-c", SYNC % ROOT], env=env, capture_output=True,
                       text=True, timeout=120)
    assert p.returncode == 0, p.stderr
    assert "RC -4 FIRST True" in p.stdout, p.stdout + p.stderr


BEHIND = r"""
import sys
sys.path.insert(0, %r)
import numpy as np
import qcs_amd
n = 14
c = qcs_amd.Circuit(n)
for t in range(10):
    c.h(t)
for t in range(10, n):
    c.x(t)
c.flush()
print("ERR", c.lib.qc_last_error(c.handle), flush=True)
want = np.zeros(1 << n)
want[15 << 10:] = 2.0 ** -5
print("OFF", float(np.max(np.abs(c.amplitudes() - want))), flush=True)
"""


def test_gates_behind_a_failed_launch_still_run(qlib):
    """Launch check 2 is the pass of the H gates, which runs and reports a
    failure; the X gates are a pass of their own behind it."""
    env = dict(os.environ, QCS_HIP_INJECT_FAULT="launch:2")
    p = subprocess.run([sys.executable, "-c", BEHIND % ROOT], env=env, capture_output=True,
                       text=True, timeout=120)
    assert p.returncode == 0, p.stderr
    assert "ERR -4" in p.stdout and p.stderr.count("injected failure") == 1, p.stdout + p.stderr
    assert float(p.stdout.split("OFF ")[1].split()[0]) <= 1e-15
