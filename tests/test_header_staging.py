"""Line headers on a HIP runtime without a device: a call on one stream does not
wait for what is queued on another's; lines of another device than the current
one are copied by the runtime, not by a kernel of this one."""
from fakehip import run


def test_streams_do_not_wait_for_each_other():
    run("""
T.init(0)
lines = [T.DeviceArray((5, 20), np.complex64) for _ in range(2)]
busy, idle = T.Stream(), T.Stream()
F.fake_block(busy.ptr, 1)
first = threading.Thread(target=T.headers_dtoh, args=(lines[0], busy), daemon=True)
first.start()
while not F.fake_waiting(busy.ptr):
    time.sleep(0.001)
second = threading.Thread(target=T.headers_dtoh, args=(lines[1], idle), daemon=True)
second.start()
second.join(10)
assert not second.is_alive(), "waits for another stream"
assert first.is_alive()
F.fake_block(busy.ptr, 0)
first.join(10)
assert not first.is_alive()
""")


def test_idle_chunks_are_bounded():
    run("""
T.init(0)
lines = T.DeviceArray((5, 20), np.complex64)
streams = [T.Stream() for _ in range(9)]
threads = [threading.Thread(target=T.headers_dtoh, args=(lines, s)) for s in streams]
for s in streams:
    F.fake_block(s.ptr, 1)
for t in threads:
    t.start()
while not all(F.fake_waiting(s.ptr) for s in streams):
    time.sleep(0.001)
for s in streams:
    F.fake_block(s.ptr, 0)
for t in threads:
    t.join(10)
calls = [c[0] for c in log()]
assert calls.count("hipHostMalloc") - calls.count("hipHostFree") <= 4
""")


def test_lines_of_another_device():
    run("""
T.init(0)
raw = np.arange(5 * 160, dtype=np.uint8).reshape(5, 160)
lines = T.DeviceArray((5, 20), np.complex64)
lines.upload(raw.view(np.complex64))
F.fake_owner(lines.ptr, 3)
assert np.array_equal(T.headers_dtoh(lines), raw[:, :80])
raw[:, :80] = 7
T.headers_htod(lines, raw[:, :80])
assert np.array_equal(lines.download().view(np.uint8).reshape(raw.shape), raw)
assert not launches(log(), "k_headers")
""")
