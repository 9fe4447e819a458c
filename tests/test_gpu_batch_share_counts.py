"""That batched circuits are shared by work-groups, and that a run whose parts
do not meet is repeated unshared: by the counts of work items and repeats the
batch reports, beside its samples."""
import numpy as np
import pytest

import qcs_amd
from qcs_amd import circuits as C

pytestmark = pytest.mark.gpu


def circuits(specs):
    cs = []
    for i, (n, d, fused) in enumerate(specs):
        c = qcs_amd.Circuit(n, qcs_amd.DEFERRED | (qcs_amd.FUSED_FP32 if fused else 0))
        c.apply(C.layered(n, d, 10 + i))
        cs.append(c)
    return cs


def sample(b, cs):
    qcs_amd.libc().srand(3)
    return b.sample(cs, 100)


# a streamed circuit of each precision alone is shared; circuits of one tile
# (13 / 14 bits) are not, and QCS_BATCH_MAX_PARTS=1 shares none
@pytest.mark.parametrize("specs,shared", [([(15, 6, True)], True), ([(14, 6, False)], True),
                                          ([(14, 6, True), (13, 6, False)], False)])
def test_streamed_circuits_are_shared(qlib, monkeypatch, specs, shared):
    cs = circuits(specs)
    with qcs_amd.Batch() as b:
        sample(b, cs)
        items, fallbacks = b.last_sharing()
        assert (items > len(cs)) == shared and fallbacks == 0
        monkeypatch.setenv("QCS_BATCH_MAX_PARTS", "1")
        cs[0].x(0)  # planned anew
        sample(b, cs)
        assert b.last_sharing() == (len(cs), 0)
    for c in cs:
        c.close()


@pytest.mark.parametrize("options", [0, qcs_amd.BATCH_GRAPH])
def test_parts_that_do_not_meet_are_repeated_unshared(qlib, monkeypatch, options):
    cs = circuits([(17, 3, False), (17, 3, True)])
    with qcs_amd.Batch(options) as b:
        want = sample(b, cs)
        assert b.last_sharing()[0] > 2
        monkeypatch.setenv("QCS_BATCH_PART_SPINS", "0")  # no patience at all
        cs[0].x(0)
        cs[0].x(0)
        again = sample(b, cs)  # planned anew
        assert b.last_sharing() == (2, 1)
    assert np.array_equal(want, again)
    for c in cs:
        c.close()


@pytest.mark.parametrize("options", [0, qcs_amd.BATCH_GRAPH])
def test_reruns_after_a_repeat_are_shared_again(qlib, monkeypatch, options):
    """A plan keeps its shares when its parts once did not meet.  While they
    keep failing to, the runs that try to share get rarer: after k failures in
    a row the next 2^(k-1) - 1 runs do not."""
    cs = circuits([(17, 3, False), (17, 3, True)])
    with qcs_amd.Batch(options) as b:
        want = sample(b, cs)
        shared = b.last_sharing()[0]
        assert shared > 2
        monkeypatch.setenv("QCS_BATCH_PART_SPINS", "0")
        cs[0].x(0)
        cs[0].x(0)
        runs = [(sample(b, cs), b.last_sharing())]  # planned anew, then reruns
        for _ in range(6):
            runs.append((sample(b, cs), b.last_sharing()))
        # tries: runs 0, 1, 3 (one left out) and 7 (three left out)
        assert [r[1] for r in runs] == [(2, k) for k in (1, 2, 2, 3, 3, 3, 3)]
        monkeypatch.delenv("QCS_BATCH_PART_SPINS")
        if options == qcs_amd.BATCH_GRAPH:  # (the captured limit of the waits)
            cs[0].x(1)
            cs[0].x(1)
        for _ in range(3):
            runs.append((sample(b, cs), b.last_sharing()))
        assert [r[1][0] for r in runs[7:]] == [shared] * 3
        assert runs[-1][1][1] == 3
    for idx, _ in runs:
        assert np.array_equal(idx, want)
    for c in cs:
        c.close()
