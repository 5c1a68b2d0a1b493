"""bench.py's JSON line is short enough for a log that keeps the end of the output: figures at six digits, the two that
the line is read for whole."""
import json

import bench


def test_short():
    line = {"value": 19142041954.198622, "ms_per_step": 150.77619933333608, "steps": 20, "vs_baseline": None,
            "config": {"kernel_ms": {"features": 71.32681234}, "members": 65536}, "extra": ["c", "d"], "ok": True}
    out = bench.short(line)
    assert out["value"] == line["value"] and out["ms_per_step"] == line["ms_per_step"]
    assert json.dumps(out["config"]) == '{"kernel_ms": {"features": 71.3268}, "members": 65536}'
    assert out["steps"] == 20 and out["vs_baseline"] is None and out["extra"] == ["c", "d"] and out["ok"] is True
    assert bench.short({"a": float("inf"), "b": 1e-300, "c": 0.0}) == {"a": float("inf"), "b": 1e-300, "c": 0.0}
