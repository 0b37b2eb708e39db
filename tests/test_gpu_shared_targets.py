"""Contexts of one batch that draw into the same page-locked buffer: every
context starts from the buffer as it was, and the last one's pixels stand, as
when their results are copied back one by one."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from conftest import OracleExecutor

pytestmark = pytest.mark.gpu

SIZES = [(700, 500), (640, 480), (700, 300)]


def _draw(L, ctx, seed):
    L.pfMakeCurrent(ctx)
    rng = np.random.default_rng(seed)
    L.pfDisable(0x10)
    L.pfClearColor(int(seed), 9, 9, 9)
    L.pfClear(3)
    L.pfBegin(2)
    for _ in range(60):
        L.pfColor4ub(*rng.integers(0, 256, 4).tolist())
        L.pfVertex3f(*[C.c_float(float(v)) for v in rng.uniform(-1, 1, 3)])
    L.pfEnd()


@pytest.mark.parametrize("shared", ["whole", "partly"])
def test_the_last_context_of_a_batch_stands(shared):
    L = pf.lib()
    L.pfdHostAlloc.restype = C.c_void_p
    L.pfdHostAlloc.argtypes = [C.c_size_t]
    L.pfdHostFree.argtypes = [C.c_void_p]
    if L.pfdInit() != 0:
        pytest.fail("no GPU: " + L.pfdLastError().decode())
    step = 0 if shared == "whole" else 101 * 4
    n = 700 * 500 * 4 + 8 * 101 * 4
    mem = L.pfdHostAlloc(n)
    buf = np.ctypeslib.as_array((C.c_uint8 * n).from_address(mem))
    want = np.full(n, 5, np.uint8)
    out = []
    with OracleExecutor():
        for k in range(8):
            w, h = SIZES[k % 3]
            px = np.full(w * h * 4, 5, np.uint8)
            ctx = C.c_void_p(L.pfCreateContext(px.ctypes.data, w, h, 7, 0))
            _draw(L, ctx, k)
            L.pfFinish()
            L.pfDeleteContext(ctx)
            out.append(px)
    ctxs = [L.pfCreateContext(mem + k * step, *SIZES[k % 3], 7, 0) for k in range(8)]
    for run in range(3):                                          # the third with the table of the second
        buf[:] = 5
        want[:] = 5
        for k, px in enumerate(out):
            # A clear leaves pixels 0..7 as they were before the batch.
            want[k * step:k * step + len(px)] = px
        for k, ctx in enumerate(ctxs):
            _draw(L, C.c_void_p(ctx), k)
        print(shared, run, flush=True)
        L.pfSubmitBatch((C.c_void_p * len(ctxs))(*ctxs), len(ctxs))
        if run == 0:
            bad = np.count_nonzero(buf != want)
            assert bad == 0, f"{bad} bytes differ"
            first = buf.copy()
        # Later runs start from the first one's depths: compare them with each other.
        elif run == 1:
            second = buf.copy()
        else:
            assert np.array_equal(buf, second)
    assert np.count_nonzero(first != 5) > n // 2
    for ctx in ctxs:
        L.pfMakeCurrent(C.c_void_p(ctx))
        L.pfDeleteContext(C.c_void_p(ctx))
    L.pfMakeCurrent(None)
    L.pfdHostFree(mem)
