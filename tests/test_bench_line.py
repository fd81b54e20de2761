"""The line that bench.py prints stays short enough to be read through a buffer of a few kilobytes."""
import json

import bench


def test_rows_per_call_are_short():
    entry = {
        "config": "c4x16", "op": "sasaw", "dtype": "float64", "function": "forward", "device_us": 1234.567, "bound": "mfma",
        "frac": 0.1234, "copy_us": 1234.567, "frac_of_copy": 0.123, "shape": {"A": [1000000, 9]}, "timed": "hip-graph replay",
    }  # fmt: skip
    row = bench.short_row(entry)
    assert row == ["c4x16 sasaw f64 forward", 1234.567, "mfma", 0.1234, 1234.567, 0.123]
    # sixteen calls at the sizes of the headline step and eighteen at larger ones, and what surrounds them
    assert len(json.dumps([row] * 34)) + 3500 < 8000
