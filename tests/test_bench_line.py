"""bench.py's JSON line stays short: the long tables go elsewhere, and nothing is dropped."""

from __future__ import annotations

import json

import bench


def test_tables_leave_the_line():
    row = {"proj": "gate_up", "N": 28672, "K": 4096, "M": 2048, "us": 378.84, "GB/s": 503.6, "TFLOP/s": 1269.7}
    result = {"metric": bench.METRIC, "value": 3634.4, "config": {"M": 1}, "roofline": {"achieved": 4686.3},
              "e2e": {"decode_step_ms": 2.991}, "shapes": [row] * 36, "bits_sweep": [row] * 15,
              "engine_config": [row] * 12, "cpu_baseline": {"value": 1.5, "configs": [row] * 60}}
    kept = json.dumps(result)
    line, details = bench.split_result(result)
    assert json.dumps(result) == kept  # the input is left alone
    assert line["value"] == 3634.4 and line["cpu_baseline"] == {"value": 1.5} and "shapes" not in line
    assert len(json.dumps(line)) < 600
    assert {**line, **{k: details[k] for k in ("shapes", "bits_sweep", "engine_config")},
            "cpu_baseline": {**line["cpu_baseline"], "configs": details["cpu_baseline_configs"]}} == result
    assert bench.split_result({"metric": "m", "cpu_baseline": None}) == ({"metric": "m", "cpu_baseline": None}, {})
