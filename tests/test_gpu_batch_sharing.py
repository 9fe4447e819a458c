"""Batched circuits shared by several work-groups, complex64 among them: a
batch of a few streamed circuits uses the whole device, and gives what one
work-group per circuit gives (QCS_BATCH_MAX_PARTS=1): the same operations on
the same tiles, so amplitudes and samples are equal bit for bit."""
import numpy as np
import pytest

import qcs_amd
from qcs_amd import circuits as C

pytestmark = pytest.mark.gpu


# 15 / 14: the smallest streamed complex64 / complex128 circuits (two tiles);
# one circuit alone, and more circuits than fit at once as parts
@pytest.mark.parametrize("specs", [[(15, 6, True)], [(14, 6, False)], [(19, 4, True)],
                                   [(18, 5, True), (18, 5, False), (16, 9, True), (15, 3, False),
                                    (12, 4, True), (10, 5, False)],
                                   [(17, 3, i % 2 == 0) for i in range(40)]])
def test_shared_circuits_equal_unshared(qlib, monkeypatch, specs):
    libc = qcs_amd.libc()
    res = []
    for cap in ("1", None):
        if cap:
            monkeypatch.setenv("QCS_BATCH_MAX_PARTS", cap)
        else:
            monkeypatch.delenv("QCS_BATCH_MAX_PARTS")
        cs = []
        for i, (n, d, fused) in enumerate(specs):
            c = qcs_amd.Circuit(n, qcs_amd.DEFERRED | (qcs_amd.FUSED_FP32 if fused else 0))
            c.apply(C.layered(n, d, 10 + i))
            cs.append(c)
        with qcs_amd.Batch(qcs_amd.BATCH_KEEP_STATES) as b:
            libc.srand(7)
            idx = b.sample(cs, 64)
            amps = [b.amplitudes(i, n) for i, (n, _, _) in enumerate(specs)]
        res.append((idx, amps))
        for c in cs:
            c.close()
    assert np.array_equal(res[0][0], res[1][0])
    for x, y in zip(res[0][1], res[1][1]):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("options", [0, qcs_amd.BATCH_GRAPH])
def test_parts_that_do_not_meet(qlib, monkeypatch, options):
    """With no patience at all at the pass boundaries the parts give up, every
    work-group exits, and the run is repeated with a work-group per circuit."""
    libc = qcs_amd.libc()
    cs = []
    for i, fused in enumerate((False, True)):
        c = qcs_amd.Circuit(17, qcs_amd.DEFERRED | (qcs_amd.FUSED_FP32 if fused else 0))
        c.apply(C.layered(17, 3, 30 + i))
        cs.append(c)
    with qcs_amd.Batch(options) as b:
        libc.srand(3)
        want = b.sample(cs, 100)
        monkeypatch.setenv("QCS_BATCH_PART_SPINS", "0")
        libc.srand(3)
        again = b.sample(cs, 100)  # a rerun of the plan
        cs[0].x(0)
        cs[0].x(0)                 # planned anew
        libc.srand(3)
        anew = b.sample(cs, 100)
    assert np.array_equal(want, again) and np.array_equal(want, anew)
    for c in cs:
        c.close()
