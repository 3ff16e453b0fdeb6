"""The aperture fit's reciprocal divisions and its Hermite interpolation split
over four lanes, on the host (tests/fit_division_check.cpp): equal to plain
division and to the whole interpolation bit for bit, since the fit's aperture
centres are integers."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_split_hermite_equals_whole(tmp_path):
    exe = str(tmp_path / "fit_division_check")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", "-x", "hip",
                    os.path.join(HERE, "fit_division_check.cpp"), "-o", exe],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
