"""Infinite samples through the FP64 kernel, against the oracle: a pixel whose
pulses hold one is infinite or NaN as the sum over its pulses one by one makes
it, component by component; a sample pair whose difference overflows FP32 (but
not its lerp) and NaNs outside a pixel's window change nothing else."""
import numpy as np
import pytest

from srg_amd import synth
from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [None, 1, 5, 11])
def test_infinite_samples(gpu, oracle, variant):
    sc = synth.make_burst(300, 3000, 131, 70, aperture=128, dem="fbm", seed=9, ntargets=1,
                          dem_source=synth.fbm_surface((256, 256), seed=3, hmax=400.0))
    g = sc.geom
    data = synth.host_samples(sc)
    clean, _, _, coef, azoff = oracle.backproject(g, data, sc.satloc, sc.dem)
    mid = g.S // 2
    with np.errstate(all="ignore"):
        parts = data.view(np.float32).reshape(g.L, g.S, 2)
        parts[120, mid - 40:mid - 20, 0] = np.inf
        parts[150, mid + 10:mid + 30, 1] = -np.inf
        parts[150, mid + 20:mid + 40, 0] = np.inf
        parts[171, mid - 30:mid + 15, 0] = -np.inf
        parts[200, mid + 60, 1] = np.nan
        parts[90, mid + 80:mid + 84, 0] = np.float32(3e38) * np.array([1, -1, 1, -1])
        want = oracle.backproject(g, data, sc.satloc, sc.dem)[0]
    d = [T.DeviceArray.from_host(x) for x in (data, sc.satloc, sc.dem, coef)]
    out = T.DeviceArray(want.shape, np.complex64)
    T.backproject(g, T.samples(d[0]), d[1], d[2], out, T.PLAIN_FP64, d_coef=d[3],
                  variant=variant)
    T.sync()
    a, b = (x.view(np.float32).reshape(-1) for x in (out.download(), want))
    assert np.isposinf(b).any() and np.isneginf(b).any() and np.isnan(b).any()
    np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
    np.testing.assert_array_equal(np.isposinf(a), np.isposinf(b))
    np.testing.assert_array_equal(np.isneginf(a), np.isneginf(b))
    m = np.isfinite(a) & np.isfinite(b)
    huge = m & (np.abs(b) > 1e30)
    assert huge.any()
    for k in (huge, m & ~huge):   # 1e-6 each in phase and amplitude, as elsewhere
        x, y = a[k].astype(np.float64), b[k].astype(np.float64)
        assert np.sqrt(np.sum((x - y) ** 2) / np.sum(y ** 2)) <= 2e-6
