"""The fused MD step's staged x3-neighbours for any fastest extent
(src/gauge/utils.h:110-139 staple links; su3_dev.h halo_slots / halo_site).
Host only: the check is compiled with hipcc for the host and runs every site of
lattices with L3 = 2 .. 140."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")
def test_halo_slots(tmp_path):
    exe = str(tmp_path / "halo_slots")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950",
                    os.path.join(ROOT, "tests", "halo_slots.cpp"), "-o", exe],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert " 0 wrong" in r.stdout
