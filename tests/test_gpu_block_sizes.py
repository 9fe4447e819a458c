"""The one-block-per-pass kernel at the sizes where its work-groups change.

Every launch variant and tile size adds the same products in the same order,
so the states are equal bit for bit; against an FP64 state the error is that
of FP32 arithmetic."""
import numpy as np
import pytest

import qcs_amd
from qcs_amd import circuits as C

pytestmark = pytest.mark.gpu


def fused_state(hip, n, k, variant, ops):
    with qcs_amd.Circuit(n, qcs_amd.FUSED_FP32 | qcs_amd.FUSE_K(k)) as c:
        if variant is not None:
            st = c.device_state
            for w in range(1, 6):
                assert hip.qcs_hip_set_tuning(st, 8 + w, variant) == 0
        c.apply(ops)
        return c.amplitudes()


# 10, 11: the smallest matrix-core states; 12, 13: the first larger tiles;
# 20 / 21: one-wave tiles end
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n", [10, 11, 12, 13, 20, 21])
def test_default_work_groups(qlib, n, k):
    hip, _ = qlib
    ops = C.random_circuit(n, 60, 31 * n + k)
    got = fused_state(hip, n, k, None, ops)
    with qcs_amd.Circuit(n) as p:
        p.apply(ops)
        want = p.amplitudes()
    # 60 gates at most as many blocks, each within a few FP32 roundings
    assert np.max(np.abs(got - want)) <= 60 * 4 * 2.0 ** -24
    for variant in (0, 1):
        assert np.array_equal(got, fused_state(hip, n, k, variant, ops)), variant


@pytest.mark.parametrize("n", [24, 25])
def test_line_to_the_largest_work_groups(qlib, n):
    ops = C.layered(n, 1, 5)
    with qcs_amd.Circuit(n, qcs_amd.FUSED_FP32) as f, qcs_amd.Circuit(n) as p:
        f.apply(ops)
        p.apply(ops)
        omf, mx = f.compare_with(p)
        assert omf <= 1e-11 and mx <= 1e-6
