"""Grover rounds (one reduction, a recurrence for the sums, one update)
against the rounds one after another in 64 bits, from states that are not
uniform.  The recurrence and the loop round differently by about 1e-16 a
round; a complex64 state is rounded once, by 2^-24 of an amplitude."""
import numpy as np
import pytest

import qcs_amd

pytestmark = pytest.mark.gpu


def rounds(a, m, k):
    a = a.astype(np.complex128)
    for _ in range(k):
        if m >= 0:
            a[m] = -a[m]
        a = 2.0 * a.mean() - a
    return a


@pytest.mark.parametrize("option,tol", [(qcs_amd.PLAIN_FP64, 1e-13), (qcs_amd.PLAIN_FP32, 2e-7)])
@pytest.mark.parametrize("n", [1, 2, 8, 10, 13, 19])
def test_rounds_from_any_state(qlib, n, option, tol):
    hip, _ = qlib
    rng = np.random.default_rng(n)
    N = 1 << n
    v = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    v = (v / np.linalg.norm(v)).astype(np.complex64).astype(np.complex128)
    with qcs_amd.Circuit(n, option) as c:
        for m, k in ((0, 1), (N - 1, 2), (N // 3, 7), (N // 2, 100), (-1, 1), (-1, 4)):
            c.set_amplitudes(v)
            assert hip.qcs_hip_grover(c.device_state, m, k) == 0
            want = rounds(v, m, k)
            assert np.max(np.abs(c.amplitudes() - want)) <= tol, (m, k)


def test_infinite_and_nan_amplitudes_spread(qlib):
    hip, _ = qlib
    with qcs_amd.Circuit(8) as c:
        for bad in (np.inf, np.nan):
            for at in (3, 77):  # the marked one, another one
                v = np.full(256, 0.0625, np.complex128)
                v[at] = bad
                c.set_amplitudes(v)
                assert hip.qcs_hip_grover(c.device_state, 3, 2) == 0
                assert np.all(np.isnan(c.amplitudes().real))
