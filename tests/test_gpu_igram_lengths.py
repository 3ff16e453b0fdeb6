"""GPU tests of the fused interferogram kernels at every transform length
(1024 to 8192 points) and at the widths on either side of a change of length:
against the FP64 oracle, with output lines for the one-pass kernels and too few
for them."""
import numpy as np
import pytest

from oracle import igram_oracle as IO
from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.sqrt(np.sum(np.abs(a - b) ** 2) / np.sum(np.abs(b) ** 2)))


@pytest.mark.parametrize("width,rows,looks", [
    (512, 40, (1, 1)), (513, 40, (1, 1)), (1024, 130, (4, 2)), (1025, 45, (1, 1)),
    (1789, 261, (4, 2)), (2048, 195, (3, 1)), (1500, 41, (5, 8)), (4097, 30, (1, 1)),
    (4100, 133, (4, 2)), (8192, 20, (1, 1)), (8192, 64, (7, 1)), (5000, 25, (1, 5)),
    (8193, 20, (2, 2)), (700, 1, (700, 1))])
def test_lengths(gpu, width, rows, looks):
    rng = np.random.default_rng(width + rows)
    a = (rng.standard_normal((rows, width)) + 1j * rng.standard_normal((rows, width))).astype(
        np.complex64)
    b = (0.6 * a + 0.8 * (rng.standard_normal(a.shape) + 1j * rng.standard_normal(a.shape))
         ).astype(np.complex64)
    a[:rows // 3, :width // 4] = 0
    b[rows - rows // 4:, width // 2:] = 0
    la, ld = looks
    ig, am = T.crossmul(T.DeviceArray.from_host(a), T.DeviceArray.from_host(b), scale=1e-3,
                        looksac=la, looksdn=ld)
    T.sync()
    gi, ga = ig.download(), am.download()
    oi, oa = IO.crossmul(a, b, scale=1e-3, looksac=la, looksdn=ld)
    assert gi.shape == oi.shape == (rows // ld, width // la)
    np.testing.assert_array_equal(gi == 0, oi == 0)
    # The kernels' FP32 against the oracle's FP64: as in the tests at 4096 points.
    assert rel(gi, oi) < 1e-5 and rel(ga, oa) < 1e-5, (rel(gi, oi), rel(ga, oa))
