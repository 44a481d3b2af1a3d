"""bench.py's line: the contract's fields, and no rate of operations formed from counted iterations
(whole periods of exact cycles are counted without being run)."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _keys(d):
    for k, v in d.items():
        yield k
        if isinstance(v, dict):
            yield from _keys(v)


def test_line():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    print("bench line: net86, 4096 particles", flush=True)
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--n", "4096", "--steps", "1", "--warmup", "1",
                        "--max-iter", "200", "--no-cpu"], capture_output=True, text=True, timeout=100, cwd=ROOT)
    assert r.returncode == 0, r.stderr[-2000:]
    line = json.loads(r.stdout.strip().splitlines()[-1])
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config"):
        assert k in line, k
    assert line["n_gpus"] == 1 and line["steps"] == 1 and line["value"] > 0
    assert line["config"]["fp64"]["counted_newton_iters_per_step"] > 0
    bad = {"achieved", "frac", "achieved_tflops", "iteration_latency_us", "newton_iters_per_s"}
    assert not bad & set(_keys(line)), bad & set(_keys(line))
