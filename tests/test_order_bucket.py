"""Places in an ordered call: the rule (host check, CPU only), and that what it is given leaves cold
dense particles out."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_order_bucket(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path / "order_bucket")
    subprocess.run([cxx, "-O1", "-std=c++17", "-o", exe, os.path.join(ROOT, "tests", "cpp", "order_bucket.cpp")],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]


def test_the_key_looks_at_the_temperature():
    src = open(os.path.join(ROOT, "sph-exa-nnet_amd", "csrc", "nnet_solver.hip")).read()
    key = re.search(r"int order_key\(.*?\n}", src, re.S).group(0)
    assert re.search(r"order_bucket\(.*rho\[i\] >= k::denseRho && temp\[i\] > k::minTemp\)", key), key
