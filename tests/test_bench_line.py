"""The benchmark's JSON line: the contract's fields, and short enough to be read from the output's last 8 KB."""
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import bench  # noqa: E402


def test_the_line_holds_the_contract_and_fits_the_tail():
    fields = {k: 1.25 for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step",
                                "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "attn_fwd_bwd_ms",
                                "edge_build_ms")}
    table = {f"kernel_{i}": {"avg_ms": 0.12345, "launches": 20, "traffic_bytes": 123456789} for i in range(60)}
    rec = {**fields, "config": {"workload": "w" * 150, "note": "n" * 400}, "value_basis": "b" * 350,
           "attention": {"a": "x" * 300}, "builder": {"rw_edges_per_s": 5.0, "rest": "y" * 300},
           "roofline": {"kernel": "k", "bound": "hbm", "achieved": 1.0, "peak": 8000.0, "unit": "GB/s", "frac": 0.5,
                        "frac_of_floor": 0.9, "basis": "z" * 600},
           "gather_floor": {"basis": "g" * 1200}, "kernels": table, "cpu_baseline": {"value": 2.5, "sample": "s" * 300}}
    full = {**rec, "extra_configs": [rec, rec, rec]}
    line = bench.brief(full)
    assert len(json.dumps(full)) > 8000 > 6000 > len(json.dumps(line))
    assert set(fields) | {"config", "roofline", "extra_configs"} <= set(line)
    assert all(line[k] == v for k, v in fields.items())
    for extra in line["extra_configs"]:
        assert extra["workload"] == "w" * 150 and extra["value"] == 1.25 and extra["roofline"]["frac_of_floor"] == 0.9
        assert extra["rw_edges_per_s"] == 5.0 and extra["cpu_baseline"] == 2.5
    assert "extra_configs" not in bench.brief(rec) and full["kernels"] is table
