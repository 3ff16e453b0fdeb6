"""The aperture fit with the orbit in the kernel's arguments (up to 32 state
vectors) and uploaded (more): parabolas equal to the oracle's exactly on either
side of the limit, and the image of a call that fits by itself equal to one
given those parabolas bit for bit, with the host orbit overwritten as soon as
the call returns."""
import numpy as np
import pytest

from srg_amd import synth
from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vectors", [4, 11, 32, 33, 200])
def test_fit_orbit_sizes(gpu, oracle, vectors):
    sc = synth.make_burst(260, 2600, 70, 33, aperture=100, dem="fbm",
                          dem_source=synth.fbm_surface((128, 128), seed=2, hmax=500.0),
                          ntargets=1, seed=4)
    g = sc.geom
    orbit = synth.make_orbit(35.0, -118.0, 43200.0, seed=4)
    g.timeorbit, g.xx, g.vv = orbit.state_vectors(g.tmid, vectors, 400.0 / vectors)
    coef = oracle.backproject(g, synth.host_samples(sc), sc.satloc, sc.dem)[3]
    data, sat, dem = (T.DeviceArray.from_host(x)
                      for x in (synth.host_samples(sc), sc.satloc, sc.dem))
    d_coef = T.DeviceArray((g.nlines, 3), np.float64)
    T.fit_aperture(g, dem, d_coef)
    np.testing.assert_array_equal(d_coef.download(), coef)
    out = [T.DeviceArray((g.nlines, g.demwidth), np.complex64) for _ in range(2)]
    T.backproject(g, T.samples(data), sat, dem, out[0], T.MIXED, d_coef=d_coef)
    gc = g.to_c()
    T.check(T.lib().tdbp_backproject(gc, T.samples(data), sat.ptr, dem.ptr, None, out[1].ptr,
                                     T.MIXED, None))
    for a in g._keep:
        a[:] = np.nan
    T.sync()
    a, b = (o.download() for o in out)
    assert np.any(a != 0)
    np.testing.assert_array_equal(a, b)
