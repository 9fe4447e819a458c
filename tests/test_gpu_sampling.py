"""Sampling: few shots run a work-group each, many a wave each; the same
uniforms give the same indices, whatever the size of the state, and both
follow the definition of the blockwise CDF (rows of 64, chunks of 4096)."""
import ctypes

import numpy as np
import pytest

import qcs_amd
from qcs_amd import circuits as C

pytestmark = pytest.mark.gpu


def sample(hip, state, u):
    u = np.ascontiguousarray(u)
    idx = np.full(u.size, -7, np.int64)
    assert hip.qcs_hip_sample(state, u.size, u.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                              idx.ctypes.data_as(ctypes.POINTER(ctypes.c_long))) == 0
    return idx


def scan(x):
    """Inclusive sums over the last axis in the wave's order."""
    d = 1
    while d < x.shape[-1]:
        y = x.copy()
        y[..., d:] = x[..., d:] + x[..., :-d]
        x, d = y, 2 * d
    return x


def cdf(p):
    """Cumulative probabilities as the library defines them (n >= 6); the
    chunks' chain left to right holds for up to 1024 chunks."""
    rows = p.reshape(-1, min(p.size, 4096) // 64, 64)
    s = scan(rows)
    running = np.zeros((rows.shape[0], rows.shape[1] + 1))
    for r in range(rows.shape[1]):
        running[:, r + 1] = running[:, r] + s[:, r, 63]
    excl = np.concatenate([[0.0], np.cumsum(running[:, -1])[:-1]])
    return excl[:, None, None] + (running[:, :-1, None] + s), excl + running[:, -1]


@pytest.mark.parametrize("option", [qcs_amd.PLAIN_FP64, qcs_amd.PLAIN_FP32])
@pytest.mark.parametrize("n", [1, 3, 6, 8, 11, 12, 13, 18, 23])
def test_few_and_many_shots_agree(qlib, n, option):
    hip, _ = qlib
    rng = np.random.default_rng(n)
    a = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    a[rng.random(1 << n) < 0.6] = 0.0  # zero amplitudes are never drawn
    a[-1] = 0.0
    a[0] += 1.0
    a /= np.linalg.norm(a)
    u = rng.random(9000)
    u[:4] = [0.0, np.nextafter(1.0, 0), 0.5, 1.5]
    with qcs_amd.Circuit(n, option) as c:
        c.set_amplitudes(a)
        amps = c.amplitudes()
        p = amps.real * amps.real + amps.imag * amps.imag
        total = p.sum()
        many = sample(hip, c.device_state, u)
        few = np.concatenate([sample(hip, c.device_state, x)
                              for x in np.split(u, [1, 2, 777, 777 + 4096, 8800])])
        assert np.array_equal(few, many)
        assert many[3] == -1 and few[3] == -1
        drawn = many[(u < total * (1 - 1e-9))]
        assert drawn.min() >= 0 and p[drawn].min() > 0.0
        if 6 <= n <= 18:
            table, ends = cdf(p)
            # uniforms at and next to every kind of seam
            at = rng.integers(0, 1 << n, 600)
            seams = np.concatenate([table.reshape(-1)[at], table[:, -1, -1], ends])
            seams = np.concatenate([seams, np.nextafter(seams, 0), np.nextafter(seams, 1)])
            got = np.concatenate([sample(hip, c.device_state, x)
                                  for x in np.array_split(seams, seams.size // 2048 + 1)])
            chunk = np.searchsorted(ends, seams, side="right")
            flat = table.reshape(ends.size, -1)
            prob = p.reshape(ends.size, -1)
            for g, k, x in zip(got, chunk, seams):
                if k == ends.size:
                    assert g == -1
                    continue
                hit = np.nonzero((flat[k] > x) & (prob[k] > 0.0))[0]
                want = hit[0] if hit.size else np.nonzero(prob[k] > 0.0)[0][-1]
                assert g == k * prob.shape[1] + want


def test_states_that_are_not_numbers(qlib):
    hip, _ = qlib
    n = 14
    a = np.full(1 << n, 2.0 ** (-n / 2), complex)
    u = np.random.default_rng(1).random(9000)
    with qcs_amd.Circuit(n) as c:
        for at, bad in ((5000, np.nan), (70, np.inf), (16383, np.nan)):
            b = a.copy()
            b[at] = bad
            c.set_amplitudes(b)
            many = sample(hip, c.device_state, u)
            assert np.array_equal(sample(hip, c.device_state, u[:500]), many[:500])
        c.set_amplitudes(np.zeros(1 << n, complex))
        assert (sample(hip, c.device_state, u[:3]) == -1).all()
