"""The bench's line: every key that a reader of the result takes, in a few kB."""

import json


def test_the_line_is_short_and_keeps_what_identifies_the_result():
    import bench
    contract = ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline",
                "dtype", "data", "config", "path", "errors", "roofline", "setup_s")
    record = {k: {"text": "x" * 200} if k in ("config", "errors", "roofline") else 1.25 for k in contract}
    leg = {"steps_per_s": 100.0, "ms_per_step": 10.0, "captured_steps": 0, "velocity_solver": "pcg", "autotuned": True,
           "iters": {"tentative": 11.2, "pressure": 16.0, "final": 12.2},
           "shape": {f"shape_{i}": [512, 512, 128] for i in range(60)},
           "instances_detail": [{"pressure_dofs": i, "radius": 0.1570, "peak": 0.5, "re": 99.3} for i in range(60)]}
    for name in bench.LEGS:
        record[name] = dict(leg)
    record["kernels"] = {f"kernel_{i}": {"avg_ms": 0.1, "bytes": 1e8, "GBps": 4e3} for i in range(100)}
    record["fp64_mcgs"] = None  # a path that was not run
    assert len(json.dumps(record)) > 26_000
    line = json.dumps(bench.short_record(record))
    assert len(line) < 6_000
    got = json.loads(line)
    assert all(got[k] == record[k] for k in contract) and "kernels" not in got and got["fp64_mcgs"] is None
    assert got["mixed"]["ms_per_step"] == 10.0 and got["mixed"]["iters"] == leg["iters"] and "shape" not in got["mixed"]
