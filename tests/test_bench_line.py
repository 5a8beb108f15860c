"""bench.py's result line: short enough to be read whole from the end of the
output, with every key of its contract."""
import json

import bench


def test_result_line_is_short_and_whole():
    rows = [{"shape": "Polyhedron", "query": "dist_out_normal", "n": 4194304, "avg_us": 498.336, "gbs": 690.2}] * 80
    inner = {"value": 1.0, "ms_per_step": 2.0, "p50_ms": 0.1, "p99_ms": 0.2, "per_kernel": rows, "rates": {"1/s": rows}}
    line = {"metric": "m", "value": 94.1, "unit": "Gqueries/s", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 2.1,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f64", "data": "synthetic",
            "config": {"model": "zoo", "global_batch": 1, "parallelism": "dp1"}, "roofline": {"share": 0.3},
            "forms_gqps": {"a": 1.0}, "batched": dict(inner), "mixed": {"fp64": dict(inner), "policy": "p"},
            "nav": {"value": 10.0, "mixed": dict(inner, identical_to_fp64=True)}, "serve": {"rates": {"1/s": inner}},
            "boolean": dict(inner), "per_kernel": rows}
    out = bench.summary(line)
    assert len(json.dumps(out)) < 2000 < len(json.dumps(line))
    for key in list(line)[:15]:
        assert out[key] == line[key]
    assert out["mixed"] == {"fp64": {k: inner[k] for k in ("value", "ms_per_step", "p50_ms", "p99_ms")}, "policy": "p"}
    assert out["nav"]["mixed"]["identical_to_fp64"] is True and "per_kernel" not in out
