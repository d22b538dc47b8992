"""The bench's result line stays short however many candidates the autotuner measures."""
import json
import os
import sys
from types import SimpleNamespace

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


def test_candidates_of_the_line(tmp_path):
    import bench

    log = [{"opts": {"skin": 0.1, "sub": 2, "lanes": k, "waves_per_cu": 32, "headroom": 1.25}, "pass_ms": 1.0 * k,
            "step_ms": float((k * 37) % 101), "steps_between": 3, "entries": 1 << 30} for k in range(100)]
    log.append({"opts": {}, "rejected": "too many cells", "step_ms": None})
    out = bench.candidates(SimpleNamespace(candidates=str(tmp_path)), "run", log)
    assert out["candidates_measured"] == 101
    assert [c["step_ms"] for c in out["best_candidates"]] == sorted(c["step_ms"] for c in log[:-1])[:4]
    assert len(json.dumps(out)) < 1500
    assert json.load(open(tmp_path / "candidates_run.json")) == log
    assert bench.candidates(SimpleNamespace(candidates=""), "run", "options given") == {"candidates": "options given"}
