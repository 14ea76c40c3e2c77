"""bench.py's line on stdout stays short enough for a log that keeps its last few KB, whatever the other workloads report."""
import argparse
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


def test_the_line_on_stdout_is_short_and_whole():
    import bench
    record = lambda unit: {"workload": "w" * 200, "value": 1234.5678, "unit": unit, "ms_per_step": 0.0449, "kernel_ms": 0.0447, "dtype": "f16", "kernel": "k" * 100,  # noqa: E731
                           "inputs": "i" * 250, "checked": True, "check": "c" * 250, "cpu_baseline": {"value": 1.5, "unit": unit, "cores": 16, "kind": "port", "sample": "s" * 250},
                           "roofline": {"bound": "hbm", "achieved": 5000.0, "peak": 8000.0, "unit": unit, "frac": 0.625, "traffic": 268435456}}
    args = argparse.Namespace(steps=20, warmup=5)
    by_name = {n: dict(record("TFLOP/s"), programs={"p%d" % i: "x" * 500 for i in range(20)}) for n in ("gemm_f16", "transpose", "permute", "gemm_bf16", "f8_m16", "mlir_fixtures")}
    by_name["gelu"], by_name["f8_m4096"] = record("GB/s"), {"workload": "f8_m4096", "error": "e" * 3000, "checked": False}
    text = json.dumps(bench.summary_line(args, by_name["gelu"], by_name))
    assert len(text) < 6000 and "\n" not in text
    line = json.loads(text)
    assert {"metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "config"} <= set(line)
    assert line["value"] == 1234.57 and line["steps"] == 20 and line["config"]["kernel_ms"] == 0.0447
    assert set(line["config"]["configs"]) == {"C1", "C2", "C3a", "C3b", "C4", "C5_M16", "C5_M4096"} and not line["config"]["configs"]["C5_M4096"]["checked"]
