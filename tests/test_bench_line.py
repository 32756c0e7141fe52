"""The result line of bench.py: it holds the contract's fields and stays short
whatever was run; what stays out of it is reported beside it."""
import json

import bench


def test_result_line_is_short_and_nothing_is_lost():
    table = {f"kernel_{q}": {"bytes_per_cell": 68, "avg_launch_ms": 0.1234, "frac": 0.5} for q in range(40)}
    accuracy = {"workload": "c2", "targets_met": True, "max_w_error": 0.05, "series": list(range(2000)),
                "fields_rms": table}
    contract = {"metric": "m", "value": 1.0, "unit": "u", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 7.0,
                "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "d", "data": "synthetic",
                "config": {"cells": 1}}
    result = dict(contract, kernels_ms_per_step=table, phases_roofline=table, kernels_io_roofline=table,
                  roofline_mixed_explicit=table, next_rows=table, cpu_baseline_more=table, accuracy_1h=accuracy,
                  accuracy_1h_c1=accuracy, serving_c4={"p50_latency_s": 13.8, "fp64_rerun": table})
    line, details = bench.split_details(result)
    assert {k: line[k] for k in contract} == contract
    assert len(json.dumps(line)) < 1500
    assert line["accuracy_1h"] == {"workload": "c2", "targets_met": True, "max_w_error": 0.05}
    assert line["serving_c4"] == {"p50_latency_s": 13.8}
    for key, value in result.items():
        if key == "serving_c4":
            assert details["serving_c4_fp64_rerun"] == value["fp64_rerun"]
        else:
            assert details.get(key, line.get(key)) == value, key
