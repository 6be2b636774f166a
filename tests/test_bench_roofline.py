"""bench.py's roofline records: no kernel is credited with bytes that its timed
launches do not read."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


@pytest.mark.parametrize("k", bench.WALKS)
def test_traversal_reports_measured_traffic_only(k):
    bvh = 1.8e9  # what a BVH walk of the launch's rays reads: 9.2 TB/s at these times
    r = bench.roofline(k, 0.589, 3, bvh, 130012041)
    assert r["bvh_bytes_per_launch"] == 1800000000 and "algorithmic_bytes_per_launch" not in r
    assert r["achieved"] == pytest.approx(130012041 * 3 / 0.589e-3 / 1e9, rel=1e-3)
    assert r["frac"] == pytest.approx(r["achieved"] / bench.HBM_PEAK_GBS, rel=1e-3) and r["frac"] < 0.1
    r = bench.roofline(k, 0.589, 3, bvh, None)
    assert r["achieved"] is None and r["frac"] is None


def test_pixel_passes_report_both():
    r = bench.roofline("k_ris", 0.4, 1, 1.2e9, 1.5e9)
    assert r["bound"] == "hbm" and r["frac"] == pytest.approx(0.375) and r["frac_physical"] == pytest.approx(0.4688, rel=1e-3)
    assert bench.roofline("k_ris", 0.0, 1, 1.2e9, None)["achieved"] is None
