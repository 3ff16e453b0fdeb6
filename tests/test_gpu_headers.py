"""Line headers to and from the device: every byte of every line's 80-byte
header, the samples after it untouched; one line, many, more than one staging chunk (4096), the shortest stride."""
import numpy as np
import pytest

from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlines,stride", [(1, 10), (3, 11), (257, 40), (1201, 300), (4097, 12)])
def test_headers_round_trip(gpu, nlines, stride):
    rng = np.random.default_rng(nlines)
    raw = rng.integers(0, 256, (nlines, 8 * stride), dtype=np.uint8)
    d = T.DeviceArray((nlines, stride), np.complex64)
    d.upload(raw.view(np.complex64))
    np.testing.assert_array_equal(T.headers_dtoh(d), raw[:, :80])
    new = rng.integers(0, 256, (nlines, 80), dtype=np.uint8)
    T.headers_htod(d, new)
    got = d.download().view(np.uint8).reshape(raw.shape)
    np.testing.assert_array_equal(got[:, :80], new)
    np.testing.assert_array_equal(got[:, 80:], raw[:, 80:])
