"""The bench's roofline object (no GPU): the peak that a kernel is priced against, and
HBM traffic only from a profile of the same plan."""
import json
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


class Plan:
    flops, bytes = 1e12, 1e6

    def __init__(self, description):
        self.description = description


@pytest.mark.parametrize("description,peak", [
    ("igemm_f32x3 ProjectFrameBlockReduceSum out=256x256x256 tile=8x32 rows=2", 416.7),
    ("igemm_f32_up2x3 ProjectFrameBlockReduceSum out=256x512x512 tile=4x32 rows=2", 416.7),
    ("fa_igemm_f32x3 FilterAdjointBlockReduceSum out=44x3x3 tile=32x32", 416.7),
    ("fa_igemm_f32 FilterAdjointBlockReduceSum out=512x3x3 MB=2", bench.PEAK_FP32_TFLOPS),
    ("igemm_f32 ProjectFrameBlockReduceSum out=256x256x256 MB=2", bench.PEAK_FP32_TFLOPS),
])
def test_peak(description, peak):
    r = bench.roofline(Plan(description), 1.0, bench.PEAK_FP32_TFLOPS, "op", 1, "none.json")
    assert r["peak"] == peak


def test_traffic_is_that_of_the_plan(tmp_path, monkeypatch):
    (tmp_path / "profiles").mkdir()
    (tmp_path / "profiles" / "t.json").write_text(json.dumps({"op": {"plan": "igemm_f32 a", "hbm_bytes_per_launch": 7}}))
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.roofline(Plan("igemm_f32 a"), 1.0, 157.3, "op", 1, "t.json")["traffic"] == 7
    assert bench.roofline(Plan("igemm_f32x3 a"), 1.0, 157.3, "op", 1, "t.json")["traffic"] is None
