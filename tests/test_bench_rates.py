"""bench.py's rates of the plain form from the kernel classes' totals: nothing
is reported for a class without launches, and the form as a whole counts the
gate passes."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_a_class_without_launches_has_no_rate():
    r = bench.plain_rates((0.0, 0, 0.0), (0.0, 0, 0.0), (50.0, 20, 2e11), 0.0, 0.0, 0.1)
    for k in ("k_1q", "k_cu"):
        for f in ("_avg_ms", "_gbs", "_hbm_frac", "_moved_gbs", "_moved_hbm_frac"):
            assert r[k + f] is None, k + f
    assert r["gate_passes"]["avg_ms"] == 2.5
    assert r["gate_passes"]["gbs"] == pytest.approx(4000.0)
    empty = bench.plain_rates((0.0, 0, 0.0), (0.0, 0, 0.0), (0.0, 0, 0.0), 0.0, 0.0, 0.1)
    assert empty["gate_passes"]["avg_ms"] is None and empty["step_hbm_frac"] is None


def test_the_whole_form_counts_every_launch():
    # 10 ms and 4e10 bytes of single gates beside 40 ms and 1.2e11 of passes
    r = bench.plain_rates((6.0, 3, 2.4e10), (4.0, 2, 1.6e10), (40.0, 10, 1.2e11), 3e10, 3e10, 0.1)
    assert r["gate_kernels_gbs"] == pytest.approx(1.6e11 / 0.05 / 1e9)
    assert r["step_hbm_frac"] == pytest.approx(1.6e11 / 0.1 / 1e9 / bench.HBM_PEAK_GBS)
    assert r["k_1q_avg_ms"] == 2.0 and r["k_cu_gbs"] == pytest.approx(4000.0)
    assert r["k_1q_moved_gbs"] == pytest.approx(5000.0)
