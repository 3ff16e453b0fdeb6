"""Line headers by two threads on two streams at once, several staging chunks
each: every thread gets and writes its own bytes."""
import threading

import numpy as np
import pytest

from srg_amd import tdbp as T

pytestmark = pytest.mark.gpu


def test_two_threads(gpu):
    rng = np.random.default_rng(5)
    raw = [rng.integers(0, 256, (n, 8 * 12), dtype=np.uint8) for n in (9000, 8500)]
    dev = [T.DeviceArray.from_host(r.view(np.complex64)) for r in raw]
    streams = [T.Stream(), T.Stream()]
    bad = []

    def work(k):
        T.init(0)
        for i in range(5):
            if not np.array_equal(T.headers_dtoh(dev[k], streams[k]), raw[k][:, :80]):
                bad.append((k, i, "read"))
            raw[k][:, :80] += 1
            T.headers_htod(dev[k], raw[k][:, :80], streams[k])

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not bad and not any(t.is_alive() for t in threads)
    for d, r in zip(dev, raw):
        np.testing.assert_array_equal(d.download().view(np.uint8).reshape(r.shape), r)
