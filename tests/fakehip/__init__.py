"""The library's host paths on a HIP runtime without a device (fake_hip.cpp):
`run(code)` builds it, runs `code` in a process of its own in which
libsrg_tdbp.so resolves its HIP calls there, and fails if that process does.
In `code`: T is srg_amd.tdbp, F the runtime's controls (fake_*), `log()` its
calls as lists of words, `ordered(log, a, b)` whether what call a enqueued is
done before what call b enqueued starts."""
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))

HEAD = """
import ctypes as C, os, sys, threading, time
sys.path.insert(0, {root!r})
F = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)
F.fake_block.argtypes = [C.c_void_p, C.c_int]
F.fake_waiting.argtypes = [C.c_void_p]
F.fake_owner.argtypes = [C.c_void_p, C.c_int]
F.fake_cost.argtypes = [C.c_char_p, C.c_double, C.c_double]
import numpy as np
from srg_amd import synth, tdbp as T


def log():
    n = F.fake_log(None, 0)
    b = C.create_string_buffer(n + 1)
    F.fake_log(b, n + 1)
    return [l.split() for l in b.value.decode().splitlines()]


def ordered(log, a, b):
    # Forward from call a: the streams on which all later work follows it, and
    # the events that stand behind it; a host wait orders everything after it.
    after, events = {{log[a][1]}}, set()
    for i in range(a + 1, b):
        call, w = log[i][0], log[i][1:]
        if call == "hipEventRecord" and w[0] in after:
            events.add(w[1])
        elif call == "hipStreamWaitEvent" and w[1] in events:
            after.add(w[0])
        elif call == "hipDeviceSynchronize" or (call == "hipStreamSynchronize" and w[0] in after):
            return True
    return log[b][1] in after


def launches(log, part):
    return [i for i, c in enumerate(log) if c[0] == "hipLaunchKernel" and part in c[2]]
"""


def run(code, timeout=60):
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "libfake_hip.so")
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", os.path.join(HERE, "fake_hip.cpp"), "-o", so],
                       check=True, capture_output=True, timeout=120)
        r = subprocess.run([sys.executable, "-c", HEAD.format(root=ROOT, so=so) + code],
                           capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0, r.stdout + r.stderr
