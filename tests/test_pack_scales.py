"""Packing's scales do not depend on the order in which a launch's workgroups
rewrite them (tests/pack_scales_check.cpp, built with hipcc from
srg_amd/csrc/tdbp_pack.h, whose kernels read them while others write theirs)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_any_order(tmp_path):
    exe = tmp_path / "pack_scales_check"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", "-x", "hip",
                    os.path.join(HERE, "pack_scales_check.cpp"), "-o", exe],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
