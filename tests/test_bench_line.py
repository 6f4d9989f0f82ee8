"""bench.py's result line on the CPU: the contract's keys, and never longer than
what a record of the output's end keeps."""
import json

import bench


def test_result_line_is_bounded():
    out = {k: 1.0 for k in bench.CONTRACT}
    out["config"] = {"workload": "w" * 400}
    out["recon_latency_ms"] = {"p50": 1.0, "p99": 2.0}
    out["roofline"] = {"kernel": "k" * 5000}  # does not fit
    out["cpu_baseline"] = {"value": 0.5, "cores": 16}
    out["sense2d"] = {"iters_per_s": 7000.0, "kernels_us": {str(i): i for i in range(1000)}}
    out["rows"] = ["r" * 100] * 200
    line = bench.result_line(out)
    assert len(line) <= bench.LINE_MAX and "\n" not in line
    got = json.loads(line)
    assert set(bench.CONTRACT) <= set(got)
    assert got["cpu_baseline"] == out["cpu_baseline"] and got["sense2d_iters_per_s"] == 7000.0
    assert "roofline" not in got and "rows" not in got
