"""The range compression's kept tables on a HIP runtime without a device: after a
launch that failed they are made again, and the spectrum of the chirp before it
is not taken for whole."""
import pytest

from fakehip import run


@pytest.mark.parametrize("kernel,fails", [("k_os_twiddles", 0), ("k_os_spectrum", 2)])
def test_failed_launches_leave_no_tables(kernel, fails):
    run(f"kernel, fails = {kernel!r}, {fails}" + """
T.init(0)
chirp = [T.Chirp(nsamps=9000, npts=n, nvalid=9000 - n, samplefreq=64e6, startfreq=-2.8e7, ramprate=1e12)
         for n in (1000, 1200)]
lines = T.DeviceArray((3, 9010), np.complex64)


def compress(c):
    T.range_compress(lines, c, T.DeviceArray((3, c.nvalid + 10), np.complex64))


if fails:
    compress(chirp[0])
    fails -= 1
F.fake_fail(b"hipLaunchKernel", fails)
try:
    compress(chirp[1])
    raise SystemExit("a failed launch passed")
except T.TdbpError:
    pass
F.fake_clear()
compress(chirp[0])
assert len(launches(log(), kernel)) == 1, log()
""")
