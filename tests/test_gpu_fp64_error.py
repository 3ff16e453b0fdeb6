"""The FP64 kernel's error is no larger than that of the pair by pair form it
replaced: FP32 weights 1 - f and f of the two samples, a product and an FMA,
everything else in FP64, and the stored image's roundings; ranges and phases of
the exact image in 80 bits.  Both root mean squares are over the same 10000 or
more pixels, whose ratio scatters by less than 1 %; a lerp as a + f (b - a) would
make it 1.07."""
import numpy as np
import pytest

from srg_amd import synth
from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,W,A", [(460, 160, 64), (1100, 90, 720)])
def test_error_of_pair_form(gpu, oracle, L, W, A):
    nl = 160
    sc = synth.make_burst(L, 3000, W, nl, aperture=A, dem="fbm", dlon=0.0004,
                          dem_source=synth.fbm_surface((256, 256), seed=3, hmax=400.0),
                          ntargets=0, seed=4)
    g = sc.geom
    rng = np.random.default_rng(6)
    data = (rng.standard_normal((g.L, g.S)) + 1j * rng.standard_normal((g.L, g.S))).astype(
        np.complex64)
    _, _, _, coef, azoff = oracle.backproject(g, data, sc.satloc, sc.dem)
    az = azoff.reshape(nl, W)
    out = T.DeviceArray((nl, W), np.complex64)
    dev = [T.DeviceArray.from_host(x) for x in (data, sc.satloc, sc.dem, coef)]
    T.backproject(g, T.samples(dev[0]), dev[1], dev[2], out, T.PLAIN_FP64, d_coef=dev[3])
    xyz = T.DeviceArray((nl, W, 3), np.float64)   # the kernel's own pixel positions
    T.setxyz(g, dev[2], xyz)
    T.sync()

    start = np.floor(az - A // 2 + 0.5).astype(int)
    live = (az > 0) & (start >= 0) & (start + A < g.L)   # whole windows
    assert live.sum() > 10000
    x, azs = xyz.download()[live], start[live]
    exact, pair = np.zeros(len(x), complex), np.zeros(len(x), complex)

    def terms(kind, q):   # sample pairs, fraction and phase factor of pulses q
        d = x.astype(kind) - sc.satloc[q].astype(kind)
        R = np.sqrt((d * d).sum(1))
        r = (R - kind(g.rngstart)) * (kind(1) / kind(g.dmrg))
        i = np.floor(r).astype(int)
        assert R.min() >= g.rngstart and i.max() < g.S - 1
        cyc = R * (kind(2) / kind(g.wvl))
        ph = np.exp(2j * np.pi * (cyc - np.rint(cyc)).astype(float))
        return data[q, i], data[q, i + 1], (r - i).astype(float), ph

    for k in range(A):
        a, b, f, ph = terms(np.longdouble, azs + k)
        exact += (a * (1 - f) + b * f) * ph
        a, b, f, ph = terms(np.float64, azs + k)
        w0, w1 = (1 - f).astype(np.float32), f.astype(np.float32)
        lerp = np.empty(len(x), np.complex64)
        for part in ("real", "imag"):
            u, v = getattr(a, part), getattr(b, part)
            setattr(lerp, part, (u * w0).astype(np.float64) + v.astype(np.float64) * w1)
        pair += lerp * ph
    s = np.float32(1 / A)
    pair = pair.astype(np.complex64) * s

    def rms(z):
        return np.sqrt(np.mean(np.abs(z.astype(np.complex128) - exact / A) ** 2))

    got = out.download()[live]
    print(f"kernel {rms(got):.3e}, pair form {rms(pair):.3e}, image "
          f"{np.sqrt(np.mean(np.abs(exact / A) ** 2)):.3e}")
    assert rms(got) <= 1.03 * rms(pair)
