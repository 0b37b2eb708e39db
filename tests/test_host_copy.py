"""Copies between host buffers that a few threads share: whole whatever the
size and however many callers there are, and available in a child of fork(),
which has none of those threads (worker processes that record frames with an
executor of their own)."""
import os
import subprocess
import sys
import textwrap
import threading

import numpy as np

import pixelforge_amd as pf
from conftest import ROOT

COPY = """
    import ctypes as C, os, signal, sys, time
    import numpy as np
    import pixelforge_amd as pf
    L = pf.lib()
    L.pfdHostCopy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t]
    def copy(n, seed):
        a = np.random.default_rng(seed).integers(0, 256, n, np.uint8)
        b = np.zeros(n + 64, np.uint8)
        L.pfdHostCopy(b.ctypes.data, a.ctypes.data, n)
        return np.array_equal(a, b[:n]) and not b[n:].any()
    def record(n):
        # An array draw, its frame handed to an executor that drops it.
        drop = pf.EXECUTOR(lambda f, u: 0)
        L.pfxSetExecutor(C.cast(drop, C.c_void_p), None)
        px = np.zeros(64 * 64 + 16, np.uint32)
        ctx = C.c_void_p(L.pfCreateContext(px.ctypes.data, 64, 64, 7, 0))
        L.pfMakeCurrent(ctx)
        pos = np.zeros((n, 3), np.float32)
        L.pfEnable(0x100)
        L.pfVertexPointer(3, 10, 0, C.c_void_p(pos.ctypes.data))
        L.pfDrawArrays(2, 0, n)
        L.pfFinish()
        ok = L.pfGetError() == 0
        L.pfDeleteContext(ctx)
        L.pfMakeCurrent(None)
        return ok
    def wait(pid, seconds):
        end = time.time() + seconds
        while time.time() < end:
            done, status = os.waitpid(pid, os.WNOHANG)
            if done:
                return status
            time.sleep(0.02)
        os.kill(pid, signal.SIGKILL)
        os.waitpid(pid, 0)
        return "no end"
"""


def test_a_forked_child_copies_and_records():
    script = textwrap.dedent(COPY) + textwrap.dedent("""
        assert copy(1 << 20, 1)
        pid = os.fork()
        if pid == 0:
            os._exit(0 if copy(1 << 20, 2) and copy((1 << 22) + 13, 3) and record(90000) else 3)
        status = wait(pid, 30)
        assert status == 0, status
        assert copy(1 << 21, 4)
    """)
    env = dict(os.environ, PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", script], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]


def test_concurrent_copies_are_whole():
    L = pf.lib()
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        for n in (0, 1, 262143, 262144, 262145, 1048576 + 63, 3000001):
            a = rng.integers(0, 256, n + 1, np.uint8)
            b = np.zeros(n + 64, np.uint8)
            L.pfdHostCopy(b.ctypes.data_as(pf.C.c_void_p), a.ctypes.data_as(pf.C.c_void_p), pf.C.c_size_t(n))
            if not np.array_equal(a[:n], b[:n]) or b[n:].any():
                bad.append((k, n))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
