"""The work queue at the ends of its range: the position count (host check, CPU only) and the
refusal of batches it cannot count."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_queue_passes(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path / "queue_passes")
    subprocess.run([cxx, "-O1", "-std=c++17", "-o", exe, os.path.join(ROOT, "tests", "cpp", "queue_passes.cpp")],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(1 << 32) - 1, 1 << 32, 1 << 40])
def test_more_particles_than_the_queue_counts_are_refused(n):
    # refused by the host's argument checks; the arrays are never looked at
    import numpy as np
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import nnet_mi355x as nm
    ctx = nm.Context(0)
    st = nm.device_state(torch, 14, np.ones(1), np.ones(1), np.zeros((14, 1)), np.ones(1))
    b = ctx.make_batch(14, st)
    b.n = n
    print(f"refused: n={n}", flush=True)
    with pytest.raises(RuntimeError, match="particles per batch"):
        ctx.compute([b], 1e-4)
    ctx.close()
