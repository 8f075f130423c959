"""Sine, cosine, arctangent and quotient of the U(1) kernels (trig_dev.h) against the
double and long double functions, over the ranges they are used in.  Host only: the
check is compiled with hipcc for the host."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")
def test_trig(tmp_path):
    exe = str(tmp_path / "trig")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-ffp-contract=off", "--offload-arch=gfx950",
                    os.path.join(ROOT, "tests", "trig.cpp"), "-o", exe],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "0 wrong" in r.stdout
