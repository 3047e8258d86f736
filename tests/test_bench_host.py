"""Host-side checks of bench.py that need no GPU: the byte model behind the reported GB/s and the
refusal of multi-GPU runs."""
import json
import os
import subprocess
import sys

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_algorithmic_bytes_model():
    # 2 B of value + 4 bits of delta per stored entry, int32 row_ptr, the fp16 input and output vectors
    assert bench.algorithmic_bytes(0, 0, 0) == 4
    assert bench.algorithmic_bytes(8, 1, 32) == 16 + 4 + 8 + 64 + 2
    P, rows, cols = 8388720, 4096, 4096
    assert bench.algorithmic_bytes(P, rows, cols) == 2 * P + P // 2 + 4 * 4097 + 2 * 4096 + 2 * 4096
    assert bench.dense_bytes(4096, 11008) == 2 * 4096 * 11008 + 2 * 11008 + 2 * 4096


def test_more_than_one_gpu_is_refused_with_a_message():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True,
                       cwd=ROOT, timeout=300)
    assert r.returncode != 0
    assert "--gpus 1" in (r.stderr + r.stdout)


def test_result_line_fits_a_kept_log():
    # a log that keeps the last 16000 characters holds the line whole: what is measured besides the headline is summarised
    case = {"shape": "49152x12288", "density": 0.5, "dense_us": 218.03, "dense_as_gemm_us": 221.1, "dense_gbps": 5540.9,
            "macko_warm_us": 118.8, "macko_us": 122.2, "macko_gbps": 6181.0, "pct_hbm_peak": 77.3, "speedup_vs_dense": 1.784,
            "speedup_vs_best_dense": 1.784, "stream_read_us": 124.45}
    suite = {"workload": "w" * 300, "value": 1.0, "roofline": {"frac": 0.5, "traffic_source": "t" * 300}, "cases": [case] * 12}
    out = {"value": 1.0, "cases": [case] * 18, "suites": {"large": suite, "skew": suite, "fewrows": suite, "e2e": {"seconds": 1.0}},
           "config": {"e2e": {"seconds": 1.0}}, "compress": [case] * 6, "int8_values_variant": [case] * 3, "batched_product": [case] * 4}
    line = bench.result_line(out)
    assert len(line) < 14000 and "\n" not in line
    kept = json.loads(line)
    assert kept["cases"] == out["cases"] and "cases" not in kept["suites"]["large"] and kept["config"] == out["config"]
    assert out["suites"]["large"]["cases"]
