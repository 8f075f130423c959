"""The library's documented build switches (hipcc -D): each is one the sources read,
and the fused MD step compiles with every value.  Front end only (no code is
generated): a value that a kernel does not support fails here."""
import os
import re
import subprocess

import pytest

from mesh_amd import build as B

SWITCHES = ["MESH_SHARE_UPPER", "MESH_SHARE_UPPER_F64", "MESH_SHARE_PREFETCH", "MESH_SHARE_PREFETCH_F64",
            "MESH_FORCE_WAVES", "MESH_FORCE_WAVES_F32", "MESH_FORCE_WAVES_ROWS"]


def test_switches_are_read():
    src = open(os.path.join(B.CSRC, "su3_hmc.hip")).read()
    for name in SWITCHES:
        assert re.search(rf"#ifndef {name}\n", src), name


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="hipcc not found")
@pytest.mark.parametrize("share,prefetch", [(0, 0), (1, 1), (2, 0), (3, 1)])
def test_fused_step_compiles(share, prefetch):
    cmd = [B.HIPCC, *B.FLAGS, "--cuda-device-only", "-fsyntax-only", f"-DMESH_SHARE_UPPER={share}",
           f"-DMESH_SHARE_UPPER_F64={share}", f"-DMESH_SHARE_PREFETCH={prefetch}",
           f"-DMESH_SHARE_PREFETCH_F64={prefetch}", os.path.join(B.CSRC, "su3_hmc.hip")]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
