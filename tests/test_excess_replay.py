"""Host replay of the gather addressing of the split tiles and of the FP64 kernel
(tests/replay_excess_index.cpp): indices and offsets in bounds, every pulse of a
pixel's window taken once, and every index at the pair's range, for bursts small
enough for the split tiles and one of several pulse stages with odd windows."""
import os
import subprocess

import pytest

from srg_amd import synth
from test_index_replay import write_scene

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    d = tmp_path_factory.mktemp("excess")
    exe, scene = str(d / "replay_excess_index"), str(d / "scene.bin")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-fopenmp", "--offload-arch=gfx950", "-x", "hip",
                    os.path.join(HERE, "replay_excess_index.cpp"), "-o", exe],
                   check=True, capture_output=True, timeout=300)
    src = synth.fbm_surface((256, 256), seed=8, hmax=800.0)
    write_scene(scene, [
        synth.make_burst(L, S, W, nl, aperture=A, dem="fbm", dem_source=src, ntargets=0, seed=L,
                         **kw)
        for L, S, W, nl, A, kw in (
            (300, 2600, 61, 37, 120, {}), (280, 2600, 129, 66, 97, {}),
            (1100, 2600, 70, 40, 901, {}), (1400, 4000, 64, 90, 719, {}),
            (300, 12000, 40, 24, 200, dict(dlat=0.002, dlon=0.004)))])

    def run(*form):
        r = subprocess.run([exe, scene, *map(str, form)], capture_output=True, text=True,
                           timeout=600)
        print(form, r.stdout.strip())
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_split_tiles(replay):
    replay("split")


@pytest.mark.parametrize("rows,stack", [(4, 0), (4, 1), (4, 2), (8, 0), (1, 1)])
def test_fp64_tiles(replay, rows, stack):
    replay("fp64", rows, stack)
