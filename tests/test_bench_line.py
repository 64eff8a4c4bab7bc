"""The benchmark's printed line: one JSON object with the headline's fields in
full, short enough (10 kB; 26 kB with every derived figure) to be read whole
from the tail of a log."""
from __future__ import annotations

import json

import bench


def rate(mlups, **more):
    return {"ms_per_step": 0.42521234567, "mlups": mlups, "achieved_gbs": 5996.840712, "roofline_frac": 0.7496051,
            "bytes_per_cell": 152, "final_mass": 16777222.3089123, "final_ke": 5249.249912, **more}


def full_record():
    top = {"metric": "D3Q19 MLUPS", "value": 39452.9, "unit": "MLUPS", "n_gpus": 1, "steps": 20, "warmup": 5,
           "ms_per_step": 0.42914319038391113, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
           "dtype": "f32", "data": "synthetic", "config": {"workload": "w" * 130, "cells": 16777216},
           "roofline": {"bound": "hbm", "achieved": 5996.8, "peak": 8000.0, "frac": 0.7496, "kernel": "k" * 300},
           "cpu_baseline": {"value": 95.893, "cores": 16, "sample": "s" * 150}}
    reactive = {f"f{k}_2048_rows{r}": {"mlups": 35665.89013841268, "achieved_gbs": 5421.215301038727,
                                       "bytes_per_cell": 152, "unfused_mlups": 30952.29238856131,
                                       "unfused_achieved_gbs": 5819.030969049526, "unfused_bytes_per_cell": 188}
                for k in (16, 32, 64) for r in range(10)}
    return {**top, "variants": {f"trt_f{k}fast_slabs": rate(39452.8997 + k) for k in range(17)},
            "configs": {"lattices": {f"D3Q19_384_mrt_f{k}fast_slabs": rate(39452.8997 + k) for k in range(56)},
                        "reactive_2d": reactive, "large": {f"D3Q19_{k}_trt_f32": rate(39321.4) for k in range(3)},
                        "shard": {f"d3q19_256x256x32_{k}": {"mlups": 35473.7613, "step_us": 59.118399620056,
                                                            "roofline_frac": 0.67400146} for k in range(8)},
                        "adjoint": {"workload": "w" * 90, "adjoint_over_forward": 2.1805325910491398}}}


def test_line_is_short_and_keeps_the_headline():
    record = full_record()
    assert len(json.dumps(record)) > 20000
    line = bench.headline(record)
    assert "\n" not in line and len(line) <= 10000
    got = json.loads(line)
    for key in record:
        if key not in ("variants", "configs"):
            assert got[key] == record[key], key
    assert list(got["variants"]) == list(record["variants"]) and list(got["configs"]) == list(record["configs"])
    assert got["variants"]["trt_f3fast_slabs"] == 39456.0
    assert got["configs"]["lattices"]["D3Q19_384_mrt_f0fast_slabs"] == 39453.0
    assert got["configs"]["reactive_2d"]["f16_2048_rows0"] == {"mlups": 35666.0, "unfused_mlups": 30952.0}
    assert got["configs"]["adjoint"]["adjoint_over_forward"] == 2.1805
