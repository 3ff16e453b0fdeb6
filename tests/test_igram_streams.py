"""The interferograms' device-wide state under several streams, on a HIP runtime
without a device: what one stream's call leaves for another's is done before it
is read."""
from fakehip import run

SETUP = """
T.init(0)
a, b = (T.DeviceArray((40, 700), np.complex64) for _ in range(2))
s1, s2 = T.Stream(), T.Stream()
"""


def test_tables_are_done_before_another_stream_reads_them():
    run(SETUP + """
T.crossmul(a, b, stream=s1)
T.crossmul(a, b, stream=s2)
l = log()
made, read = launches(l, "k_up_tables"), launches(l, "k_xmul")
assert len(made) == 4 and len(read) == 2
assert all(ordered(l, m, r) for m in made for r in read), l
""")


def test_tables_that_failed_are_made_again():
    run(SETUP + """
F.fake_fail(b"hipLaunchKernel", 2)
try:
    T.crossmul(a, b, stream=s1)
    raise SystemExit("a failed launch passed")
except T.TdbpError:
    pass
F.fake_clear()
T.crossmul(a, b, stream=s1)
assert len(launches(log(), "k_up_tables")) == 4, log()
""")
