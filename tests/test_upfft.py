"""The 1024- and 2048-point FFT pairs of the interferograms' upsampling on the
host (tests/upfft_check.cpp, built with hipcc from srg_amd/csrc/tdbp_osfft.h):
DIF within 1e-6 relative RMS of a direct long-double DFT, the pair returning N
times its input within 2e-6."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_short_pairs_against_direct_dft(tmp_path):
    exe = tmp_path / "upfft_check"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", "-x", "hip",
                    os.path.join(HERE, "upfft_check.cpp"), "-o", exe],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
