"""bench.py's output line stays short enough to be kept whole: the
records of the served requests go to stderr, not into the line."""
import json
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_request_records_stay_out_of_the_line(capsys):
    sys.path.insert(0, str(ROOT))
    import bench
    record = {"rid": 0, "body": "ellipsoid", "re": 1352202.9, "cells": 2271744, "levels": 4, "coarse_steps": 128,
              "cd_avg_fp32": 2.23388, "cd_avg_fp16": 2.234011, "status": ["ok", "ok"], "latency_fp32_s": 9.679}
    serving = {"requests": 64, "cases_per_hour_ratio": 2.34, "per_request": [dict(record, rid=i) for i in range(64)]}
    line = bench.serving_line(serving)
    assert line == {"requests": 64, "cases_per_hour_ratio": 2.34}
    err = capsys.readouterr().err
    rows = [json.loads(ln[ln.index("{"):]) for ln in err.splitlines() if "request {" in ln]
    assert rows == serving["per_request"]
    assert bench.serving_line(None) is None
