"""Page-locked memory of recorded frames: a few allocations for points and
lines, none for the array elements of a context's only frame, kept while
frames use it, given back when they no longer do or the context goes, and
bounded over all contexts.  The library's page-locked allocations are counted in a process of its own, by
functions that take hipHostMalloc's and hipHostFree's place."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = """
#include <stddef.h>
typedef int (*Malloc)(void**, size_t, unsigned);
typedef int (*Free)(void*);
static Malloc realMalloc;
static Free realFree;
static struct { void* p; size_t n; } at[4096];
static size_t total;
static int calls;
void shim_set(void* m, void* f) { realMalloc = (Malloc)m; realFree = (Free)f; }
size_t shim_total(void) { return total; }
int shim_calls(void) { return calls; }
int hipHostMalloc(void** p, size_t n, unsigned flags)
{
    const int e = realMalloc(p, n, flags);
    calls++;
    for (int k = 0; e == 0 && k < 4096; k++)
        if (!at[k].p) { at[k].p = *p; at[k].n = n; total += n; break; }
    return e;
}
int hipHostFree(void* p)
{
    for (int k = 0; k < 4096; k++)
        if (p && at[k].p == p) { total -= at[k].n; at[k].p = 0; break; }
    return realFree(p);
}
"""

SCRIPT = """
    import ctypes as C, sys
    import numpy as np
    shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    import pixelforge_amd as pf
    hip = C.CDLL(sys.argv[2])
    shim.shim_set(C.cast(hip.hipHostMalloc, C.c_void_p), C.cast(hip.hipHostFree, C.c_void_p))
    shim.shim_total.restype = C.c_size_t
    L = pf.lib()
    assert L.pfdInit() == 0, L.pfdLastError()
    drop = pf.EXECUTOR(lambda f, u: 0)                  # frames are recorded, not run
    L.pfxSetExecutor(C.cast(drop, C.c_void_p), None)
    pos = np.random.default_rng(0).uniform(-1, 1, (2000000, 3)).astype(np.float32)
    idx = np.zeros(300, np.uint32)
    keep = []
    def context():
        px = np.zeros(64 * 64 + 16, np.uint32)
        keep.append(px)
        return C.c_void_p(L.pfCreateContext(px.ctypes.data, 64, 64, 7, 0))
    def draw(kind, n):
        L.pfEnable(0x100)
        L.pfVertexPointer(3, 10, 0, C.c_void_p(pos.ctypes.data))
        if kind == "arrays":
            # Few triangles that read n elements: their host streams stay small.
            idx[0] = n - 1
            L.pfDrawElements(2, 300, 5, C.c_void_p(idx.ctypes.data))
        else:
            L.pfDrawArrays({"points": 0, "lines": 1}[kind], 0, n)
    def frame(ctx, kind, n):
        L.pfMakeCurrent(ctx)
        before = shim.shim_calls(), shim.shim_total()
        draw(kind, n)
        L.pfFinish()
        assert L.pfGetError() == 0
        return shim.shim_calls() - before[0], shim.shim_total() - before[1]
    for kind, bytes_each in (("points", 32), ("lines", 28), ("arrays", 12)):
        base = context()
        few = [frame(base, kind, 4) for _ in range(3)]  # the context's other memory
        assert few[2][0] == 0, few
        ctx = context()
        got = [frame(ctx, kind, n) for n in (100000, 100000, 100000, 90000, 1000000, 1000000, 1000000)]
        print(kind, few, got, flush=True)
        # Array elements: nothing in the first frame, one block in the second.
        # Points and lines: doubled from 128 KiB on.  Then nothing, and the
        # same where the frames get larger.
        first, second = (0, 1) if kind == "arrays" else (5, 0)
        assert few[0][0] <= got[0][0] <= few[0][0] + first
        assert got[1][0] == second
        assert 100000 * bytes_each <= got[0][1] + got[1][1] - few[0][1] <= 300000 * bytes_each
        assert got[2] == got[3] == (0, 0)
        assert got[4][0] <= first and got[5][0] == second and got[6] == (0, 0)
        held = sum(g[1] for g in got) - few[0][1]
        assert 1000000 * bytes_each <= held <= 64 << 20
        small = [frame(ctx, kind, 4) for _ in range(60)]
        assert -held <= sum(s[1] for s in small) <= 4096 - held, (held, small)
        got = [frame(ctx, kind, n) for n in (500000, 500000)]
        before = shim.shim_total()
        L.pfDeleteContext(ctx)
        assert before - shim.shim_total() >= 500000 * bytes_each
        L.pfDeleteContext(base)
    # All contexts together.
    start = shim.shim_total()
    ctxs = [context() for _ in range(40)]
    for _ in range(2):
        for c in ctxs:
            frame(c, "arrays", 1500000)                 # 18 MB and slack each
    held = shim.shim_total() - start
    print("contexts hold", held, flush=True)
    assert 300 << 20 < held <= (512 << 20) + 40 * (8 << 20)
    for c in ctxs:
        L.pfMakeCurrent(c)
        L.pfDeleteContext(c)
    print("after", shim.shim_total() - start, flush=True)
    assert shim.shim_total() <= start
"""


def test_recording_memory_is_bounded_and_given_back(tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(so)], check=True)
    r = subprocess.run([sys.executable, "-u", "-c", textwrap.dedent(SCRIPT), str(so), "/opt/rocm/lib/libamdhip64.so"],
                       cwd=ROOT, env=dict(os.environ, PYTHONPATH=ROOT), capture_output=True, text=True, timeout=100)
    print(r.stdout[-4000:], r.stderr[-3000:], flush=True)
    assert r.returncode == 0
