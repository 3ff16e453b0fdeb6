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


# Few output lines (two passes over a shared batch), a width without a fused
# kernel, and both after one another.
def test_calls_take_turns_with_the_batch_buffers():
    run(SETUP + """
wide = [T.DeviceArray((9, 8200), np.complex64) for _ in range(2)]
for stream, pair, looks in ((s1, (a, b), 8), (s2, (a, b), 8), (s1, wide, 2), (s2, (a, b), 8)):
    T.crossmul(*pair, looksdn=looks, stream=stream)
l = log()
read = launches(l, "k_xmulEPK")
write = launches(l, "k_up_fused") + launches(l, "k_up_load")
assert len(read) == 4 and launches(l, "k_up_load"), l
for r in read:
    later = [w for w in write if w > r]
    assert all(ordered(l, r, w) for w in later), l
""")


def test_buffers_of_a_graph_are_kept():
    run(SETUP + """
keep = [T.crossmul(a, b, looksdn=8, stream=s1)]
cap = C.c_void_p(s1.ptr)
F.hipStreamBeginCapture(cap, 0)
keep.append(T.crossmul(a, b, looksdn=8, stream=s1))
F.hipStreamEndCapture(cap, C.byref(C.c_void_p()))
F.fake_clear()
big = T.DeviceArray((24, 8192), np.complex64)
keep.append(T.crossmul(big, big, looksdn=12, stream=s2))
assert [c for c in log() if c[0] == "hipDeviceSynchronize"]   # they grew
assert not [c for c in log() if c[0] == "hipFree"], log()
""")
