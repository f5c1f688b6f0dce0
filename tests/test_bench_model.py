"""The ceilings that bench.py holds the U-list kernels against."""
import sys
from pathlib import Path

import pytest

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
import bench  # noqa: E402


@pytest.mark.parametrize("kind,reached", [("mixed", 80.5), ("fp64", 29.0)])
def test_no_kernel_is_above_its_issue_bound(kind, reached):
    """The rates (TFLOP/s, 11 flop a pair) the kernels have reached are below
    the bound, and the bound is below the published peak."""
    b = bench.issue_bound(kind, reached)
    assert 0.5 < b["frac"] < 1.0 and b["frac"] == reached / b["tflops"]
    assert b["tflops"] < {"mixed": bench.FP32_PEAK_TFLOPS, "fp64": bench.FP64_PEAK_TFLOPS}[kind]
    assert b["tflops"] == pytest.approx(11.0 * b["pairs_per_cycle_per_simd"] * 1024 * 2.4e9 / 1e12)
