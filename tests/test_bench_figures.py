"""The figures bench.py derives: shares of a hardware rate count the operations the
kernel executes, and HBM bytes are quoted only if they were measured on the kernels
that are timed."""
import json

import bench


def test_rate_counts_executed_operations():
    pairs = 396361728                     # far pairs of the 4096-sub-grid level
    ops_ms = pairs * bench.EXECUTED_FLOPS_PER_PAIR / (bench.FP64_VALU_PEAK_TFLOPS * 1e12) * 1e3
    # a kernel that executes its operations at the peak rate has used all of it, no more
    assert abs(bench.executed_tflops(pairs, ops_ms) / bench.FP64_VALU_PEAK_TFLOPS - 1.0) < 1e-12
    # 76 FMA, 33 MUL, 4 ADD
    assert bench.EXECUTED_FLOPS_PER_PAIR == 2 * 76 + 33 + 4 < bench.FLOPS_PER_PAIR["rho"]
    # 1.99 ms: under half of the peak
    assert 0.4 < bench.executed_tflops(pairs, 1.99) / bench.FP64_VALU_PEAK_TFLOPS < 0.5


def test_traffic_of_other_kernels_is_not_quoted(tmp_path):
    path = tmp_path / "traffic_lv_v704.json"
    path.write_text(json.dumps({"hbm_bytes_per_launch": 7, "kernel_id": "aaaa"}))
    assert bench.measured_traffic("lv", 704, "aaaa", str(tmp_path)) == 7
    assert bench.measured_traffic("lv", 704, "bbbb", str(tmp_path)) is None
    assert bench.measured_traffic("lv", 702, "aaaa", str(tmp_path)) is None
    path.write_text(json.dumps({"hbm_bytes_per_launch": 7}))
    assert bench.measured_traffic("lv", 704, "aaaa", str(tmp_path)) is None
