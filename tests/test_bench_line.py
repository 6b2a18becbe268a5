"""The line that bench.py prints: every key that is promised, in the length of a
log's tail (the progress lines share it)."""
from __future__ import annotations

import json
import os
import re

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _record():
    """The full record of the committed run."""
    text = open(os.path.join(ROOT, "profiles", "bench_1080p_steps20.md")).read()
    return json.loads(re.search(r"```json\n(.*?)\n```", text, re.S).group(1))


def test_line_is_short_and_whole():
    full = _record()
    s = bench.short_line(full)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline",
              "dtype", "data", "config"):
        assert s[k] == full[k] or k == "config"
    assert s["config"]["workload"] == full["config"]["workload"]
    assert len(json.dumps(s)) <= 1300


def test_line_without_the_further_measurements():
    full = {k: v for k, v in _record().items() if k not in ("learned", "config3", "config4", "gpu_over_cpu")}
    s = bench.short_line(full)
    assert "learned" not in s and json.dumps(s)
