"""Device allocations that fail in the middle of a call: the call returns an
error, and the next one draws its frame whole.  hipMalloc is replaced by a
function that fails once it has succeeded a given number of times (in a
process of its own, before the library is loaded); no kernel is stopped."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = """
#include <stddef.h>
typedef int (*Malloc)(void**, size_t);
static Malloc real;
static int left = -1;               /* allocations until one fails; -1: none fails */
void shim_set(void* f) { real = (Malloc)f; }
void shim_arm(int n) { left = n; }
int hipMalloc(void** p, size_t n)
{
    if (left >= 0 && left-- == 0) { *p = 0; return 2; }        /* hipErrorOutOfMemory */
    return real(p, n);
}
"""

PRELUDE = """
    import ctypes as C, sys
    import numpy as np
    shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    sys.path.insert(0, sys.argv[2] + "/tests")
    import pixelforge_amd as pf
    from conftest import OracleExecutor
    hip = C.CDLL("libamdhip64.so" if len(sys.argv) < 4 else sys.argv[3])
    shim.shim_set(C.cast(hip.hipMalloc, C.c_void_p))
    L = pf.lib()
    assert L.pfdInit() == 0, L.pfdLastError()
"""

RUN_TIMED = PRELUDE + """
    params = pf.scene(kind=pf.RANDOM_3D, width=160, height=120, ntris=4000, seed=12, depthFunc=pf.PF_LEQUAL)
    with OracleExecutor():
        want, _, err = pf.render(params, pf.LIB_PATH)
    assert err == 0
    failed = 0
    for n in range(60):
        cap = pf.capture(params)
        snap = cap.snapshot()
        cap.restore(snap)
        t = pf.PFDtimes()
        shim.shim_arm(n)
        rc = L.pfdJobRunTimed(cap.job, C.byref(t))
        shim.shim_arm(-1)
        failed += rc != 0
        for run in range(2):
            cap.restore(snap)
            assert L.pfdJobLaunch(cap.job) == 0 and L.pfdJobSync(cap.job) == 0 and L.pfdJobDownload(cap.job) == 0
            got = cap.images()[0][:want.size].reshape(want.shape)
            assert np.array_equal(got, want), (n, rc, run, np.count_nonzero(got != want))
        st = pf.PFDstats()
        assert L.pfdJobStats(cap.job, C.byref(st)) == 0 and st.clippedTriangles > 0
        cap.close()
        print("timed run, allocation", n, "rc", rc, flush=True)
        if rc == 0:
            break
    assert 10 < failed < 60
"""

BATCH = PRELUDE + """
    def context(w, h, seed):
        px = np.zeros(w * h + 16, np.uint32)
        return L.pfCreateContext(px.ctypes.data, w, h, 7, 0), px, w * h, seed
    def draw(c):
        ctx, px, n, seed = c
        L.pfMakeCurrent(C.c_void_p(ctx))
        rng = np.random.default_rng(seed)
        L.pfDisable(0x10)
        L.pfClear(3)
        L.pfBegin(2)
        for _ in range(40):
            L.pfColor4ub(*rng.integers(0, 256, 4).tolist())
            L.pfVertex3f(*[C.c_float(float(v)) for v in rng.uniform(-1, 1, 3)])
        L.pfEnd()
    big = context(300, 200, 1)
    many = [context(16 + k % 5, 16, 2 + k) for k in range(40)]
    with OracleExecutor():
        draw(big)
        L.pfFinish()
    want = big[1].copy()
    draw(big)
    L.pfFinish()
    assert np.array_equal(big[1], want)
    failed = 0
    for k in range(80):
        for c in many:
            draw(c)
        # One buffer more each time, then none.
        shim.shim_arm(1 if k else 0)
        L.pfSubmitBatch((C.c_void_p * len(many))(*[c[0] for c in many]), len(many))
        shim.shim_arm(-1)
        errors = []
        for c in many:
            L.pfMakeCurrent(C.c_void_p(c[0]))
            errors.append(L.pfGetError())
        big[1][:] = 0
        draw(big)
        L.pfFinish()
        assert L.pfGetError() == 0 and np.array_equal(big[1], want), (k, np.count_nonzero(big[1] != want))
        print("batch", k, "error", errors[0], flush=True)
        failed += errors[0] != 0
        if errors[0] == 0:
            break
    assert 3 < failed < 80
"""


@pytest.mark.parametrize("script", [RUN_TIMED, BATCH], ids=["timed_run", "batch"])
def test_the_call_after_a_failed_allocation_draws_whole(script, tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(so)], check=True)
    hip = "/opt/rocm/lib/libamdhip64.so"
    r = subprocess.run([sys.executable, "-u", "-c", textwrap.dedent(script), str(so), ROOT] + ([hip] if os.path.exists(hip) else []),
                       cwd=ROOT, env=dict(os.environ, PYTHONPATH=ROOT), capture_output=True, text=True, timeout=100)
    print(r.stdout[-3000:], r.stderr[-3000:], flush=True)
    assert r.returncode == 0
