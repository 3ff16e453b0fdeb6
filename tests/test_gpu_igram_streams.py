"""Interferograms enqueued on two streams without a wait between them, each with
its own images: looked pairs of few output lines (which share one batch of
upsampled rows), at a width with a fused kernel and one without, and a looked
pair in one pass; every result equals the one of the call by itself."""
import numpy as np
import pytest

from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,rows,looks", [(1000, 48, (2, 8)), (8300, 12, (3, 4)),
                                              (1500, 400, (4, 2))])
def test_two_streams(gpu, width, rows, looks):
    rng = np.random.default_rng(width)
    pairs = [[T.DeviceArray.from_host((rng.standard_normal((rows, width))
                                       + 1j * rng.standard_normal((rows, width))
                                       ).astype(np.complex64)) for _ in range(2)]
             for _ in range(2)]
    kw = dict(scale=1e-3, looksac=looks[0], looksdn=looks[1])
    want = []
    for p in pairs:
        want.append([x.download() for x in T.crossmul(*p, **kw)])
    streams = [T.Stream(), T.Stream()]
    T.sync()
    got = [[T.crossmul(*p, stream=s, **kw) for p, s in zip(pairs, streams)] for _ in range(10)]
    T.sync()
    for both in got:
        for outs, w in zip(both, want):
            for x, y in zip(outs, w):
                np.testing.assert_array_equal(x.download(), y)
