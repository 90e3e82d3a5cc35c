"""bench.py's command line on the CPU: more than one GPU is refused with a message (this
build measures one GPU), before anything touches a device; and the printed line keeps the
headline's keys within its length whatever the other workloads say."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused():
    out = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                         text=True, timeout=120)
    assert out.returncode == 2
    msg = json.loads(out.stdout.strip().splitlines()[-1])
    assert "one GPU" in msg["error"]


def test_printed_line_is_short():
    sys.path.insert(0, ROOT)
    import bench
    roofline = {"bound": "hbm", "achieved": 2567.123456, "peak": 8000.0, "unit": "GB/s", "frac": 0.32089,
                "kernel": "k" * 200, "valu": {"frac": 0.66}, "avg_ms": 18.5}
    cpu = {"value": 1.5871234, "unit": "mul+relin ops/s", "cores": 1, "kind": "reference", "how": "h" * 300}
    sub = {"metric": "m" * 120, "value": 33517.123456789, "unit": "rotations/s", "roofline": roofline,
           "cpu_baseline": cpu, "config": {"workload": "w" * 200}}
    out = {"metric": "HE mul+relin ops/s at N=2^16 batched vs plain; p50/p99 served latency", "value": 3256.123456,
           "unit": "mul+relin ops/s", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 39.312345678,
           "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "u64",
           "data": "synthetic (seeded uniform residues; injected uniform relinearization key)",
           "config": {"workload": "c" * 130, "parallelism": "single GPU"}, "roofline": roofline, "cpu_baseline": cpu,
           "batched_over_plain": 1.46, "plain": {"x": "y" * 400},
           "served_latency": {"batched": {"p50_ms": 0.87, "p99_ms": 3.2, "n": 5}, "rate": 3.0},
           "configs": {f"workload_number_{k}": sub for k in range(20)}}
    out["configs"]["broken"] = {"error": "RuntimeError: " + "e" * 500}
    line = bench.short_line(out)
    assert len(json.dumps(line)) <= bench.LINE_LIMIT
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config"):
        assert k in line
    assert abs(line["value"] / out["value"] - 1) < 1e-4 and line["config"] == out["config"]
    few = dict(out, configs={"chain": sub, "broken": out["configs"]["broken"]})
    assert bench.short_line(few)["configs"]["chain"] == "33517 rotations/s"
    assert bench.short_line(few)["roofline"]["frac"] == 0.32089
    assert bench.short_line(few)["served_ms"] == {"batched": {"p50_ms": 0.87, "p99_ms": 3.2}}
