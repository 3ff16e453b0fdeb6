"""Bursts with too few pixels to fill the chip, whose pulses are split over a
workgroup's waves: a batch that mixes such bursts with whole-tile ones equals
one launch per burst bit for bit; pixel counts that do not divide by the tile,
and fewer pulses in the last stage than waves, against the oracle (the bounds
of the FP64 and mixed kernels elsewhere: 1e-6 rad / 1e-6, 1 mrad / 1e-4)."""
import numpy as np
import pytest

from srg_amd import synth
from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu
SRC = synth.fbm_surface((256, 256), seed=8, hmax=800.0)


def scene(L, S, W, nl, A, seed):
    return synth.make_burst(L, S, W, nl, aperture=A, dem="fbm", dem_source=SRC, ntargets=2,
                            seed=seed)


def upload(sc):
    data = synth.host_samples(sc)
    return data, [T.DeviceArray.from_host(x) for x in (data, sc.satloc, sc.dem)]


@pytest.mark.parametrize("precision", [T.PLAIN_FP64, T.MIXED])
def test_batch_of_split_and_whole_bursts(gpu, precision):
    scenes = [scene(300, 2600, 61, 37, 120, 1), scene(420, 3400, 400, 420, 64, 2),
              scene(280, 2600, 129, 66, 96, 3)]
    batch = T.Batch(precision)
    keep, outs, singles = [], [], []
    for sc in scenes:
        d = upload(sc)[1]
        keep.append(d)
        o = [T.DeviceArray((sc.geom.nlines, sc.geom.demwidth), np.complex64) for _ in range(2)]
        outs.append(o)
        T.backproject(sc.geom, T.samples(d[0]), d[1], d[2], o[0], precision)
        batch.add(sc.geom, T.samples(d[0]), d[1], d[2], o[1])
        singles.append(o[0])
    for _ in range(2):
        batch.run()
    T.sync()
    for single, whole in outs:
        a = single.download()
        assert np.any(a != 0)
        np.testing.assert_array_equal(a, whole.download())
    batch.close()


@pytest.mark.parametrize("L,W,nl,A", [(130, 17, 5, 31), (300, 33, 9, 257), (900, 16, 6, 770)])
def test_split_matches_oracle(gpu, oracle, L, W, nl, A):
    sc = scene(L, 2600, W, nl, A, 7)
    data, d = upload(sc)
    want, _, _, _, azoff = oracle.backproject(sc.geom, data, sc.satloc, sc.dem)
    m = azoff > 0
    assert m.any()
    out = T.DeviceArray(want.shape, np.complex64)
    for precision, phase, amp in ((T.PLAIN_FP64, 1e-6, 1e-6), (T.MIXED, 1e-3, 1e-4)):
        T.backproject(sc.geom, T.samples(d[0]), d[1], d[2], out, precision)
        T.sync()
        g, o = out.download().astype(np.complex128), want.astype(np.complex128)
        assert np.all(g[~m] == 0)
        g, o = g[m], o[m]
        w = np.abs(o) ** 2
        assert np.sqrt(np.sum(w * np.angle(g * np.conj(o)) ** 2) / np.sum(w)) <= phase
        assert np.sqrt(np.sum((np.abs(g) - np.abs(o)) ** 2) / np.sum(w)) <= amp
