"""The FP64 kernel's excess form where it can go wrong, against the oracle:
windows shorter than its quartic needs (< 32 pulses), partial and odd blocks,
more pulses than one stage holds (768), tiles that leave the range gate, coarse
posting (short blocks or none), pulse positions off any smooth path (all of
them, or one between the quartic's nodes), every tile shape.

Both sides are FP64 sums of FP32 lerps (rounding ~6e-8 of a sample); range and
phase differ by 1e-10 m (2e-8 rad).  Bound as for the FP64 kernel elsewhere:
1e-6 rad, 1e-6 in amplitude."""
import numpy as np
import pytest

from srg_amd import synth
from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu

CASES = {
    "aperture-24": dict(L=200, A=24),
    "aperture-40": dict(L=200, A=40),
    "aperture-97": dict(L=300, A=97, W=65, nlines=37),
    "stages": dict(L=1100, A=900, W=96, nlines=24),
    "gate": dict(L=300, A=128, S=600, W=128),
    "coarse": dict(L=300, A=200, dlat=0.002, dlon=0.004, W=40, nlines=24, S=12000),
    "coarser": dict(L=300, A=200, dlat=0.01, dlon=0.02, W=24, nlines=20, S=24000),
    "jitter": dict(L=300, A=128, jitter=0.002),
    "one-pulse": dict(L=300, A=128, move=(171, 0.05)),
}


def errors(g, o):
    g, o = g.astype(np.complex128), o.astype(np.complex128)
    w = np.abs(o) ** 2
    return (float(np.sqrt(np.sum(w * np.angle(g * np.conj(o)) ** 2) / np.sum(w))),
            float(np.sqrt(np.sum((np.abs(g) - np.abs(o)) ** 2) / np.sum(w))))


def check(oracle, c, variants):
    sc = synth.make_burst(c["L"], c.get("S", 3000), c.get("W", 70), c.get("nlines", 48),
                          dlat=c.get("dlat"), dlon=c.get("dlon", 0.0002), aperture=c["A"],
                          dem="fbm", dem_source=synth.fbm_surface((256, 256), seed=3, hmax=400.0),
                          ntargets=2, seed=11)
    sat = sc.satloc.copy()
    if "jitter" in c:
        sat += np.random.default_rng(2).normal(0.0, c["jitter"], sat.shape)
    if "move" in c:
        sat[c["move"][0]] += c["move"][1]
    data = synth.host_samples(sc)
    want, _, _, coef, azoff = oracle.backproject(sc.geom, data, sat, sc.dem)
    m = azoff > 0
    assert m.any()
    smp = T.samples(d_data := T.DeviceArray.from_host(data))
    d_sat, d_dem = T.DeviceArray.from_host(sat), T.DeviceArray.from_host(sc.dem)
    d_coef = T.DeviceArray.from_host(coef)
    d_out = T.DeviceArray(want.shape, np.complex64)
    for v in variants:
        d_out.upload(np.full(want.shape, 7, np.complex64))
        T.backproject(sc.geom, smp, d_sat, d_dem, d_out, T.PLAIN_FP64, d_coef=d_coef, variant=v)
        T.sync()
        got = d_out.download()
        ph, amp = errors(got[m], want[m])
        print(f"variant {v}: {int(m.sum())} px, phase {ph:.2e} rad, amp {amp:.2e}")
        assert ph <= 1e-6 and amp <= 1e-6
        assert np.all(got[~m] == 0)
    assert d_data.ptr


@pytest.mark.parametrize("name", sorted(CASES))
def test_excess_form(gpu, oracle, name):
    check(oracle, CASES[name], [None, 5])


def test_every_tile_shape(gpu, oracle):
    check(oracle, dict(L=300, A=128, W=131, nlines=70), range(8))
