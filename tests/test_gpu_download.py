"""Downloads of a job's targets into host memory of every kind: page-locked
buffers at any alignment (one kernel writes them all), ordinary ones, and
both in one batch; sizes around the 16 KiB a workgroup copies.  Every pixel
must equal the oracle's and the bytes around a target must stay as they
were."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from conftest import OracleExecutor

pytestmark = pytest.mark.gpu

TARGETS = {(7, 0): 4, (6, 0): 3, (6, 2): 2, (7, 9): 8}
GUARD = 64


def _scene(ctx, seed):
    L = pf.lib()
    L.pfMakeCurrent(ctx)
    rng = np.random.default_rng(seed)
    L.pfDisable(0x10)
    L.pfEnable(0x8)
    L.pfClearColor(1, 2, 3, 4)
    L.pfClear(3)
    L.pfBegin(2)
    for _ in range(30):
        L.pfColor4ub(*rng.integers(0, 256, 4).tolist())
        L.pfVertex3f(*[C.c_float(float(v)) for v in rng.uniform(-1, 1, 3)])
    L.pfEnd()


def _frames():
    out = []
    for k, (w, h) in enumerate([(64, 64), (64, 64), (1, 1), (37, 29), (128, 33), (5, 3), (200, 41), (127, 129), (16, 256)]):
        for fmt, bpp in TARGETS.items():
            for off in (0, 1, 2, 4, 8, 16):
                if off % (2 if fmt[1] in (2, 9) else 1) == 0 and not (fmt == (7, 0) and off % 4):
                    out.append((w, h, fmt, bpp, off, (k + off) % 3 != 2))
    return out


def test_targets_of_every_kind_in_one_batch():
    L = pf.lib()
    L.pfdHostAlloc.restype = C.c_void_p
    L.pfdHostAlloc.argtypes = [C.c_size_t]
    L.pfdHostFree.argtypes = [C.c_void_p]
    frames = _frames()
    want = []
    with OracleExecutor():
        for i, (w, h, fmt, bpp, off, pinned) in enumerate(frames):
            buf = np.full(w * h * bpp + 16, 5, np.uint8)
            ctx = C.c_void_p(L.pfCreateContext(buf.ctypes.data, w, h, *fmt))
            _scene(ctx, i)
            L.pfFinish()
            L.pfDeleteContext(ctx)
            want.append(buf[:w * h * bpp])
    ctxs, bufs, allocs = [], [], []
    for i, (w, h, fmt, bpp, off, pinned) in enumerate(frames):
        n = w * h * bpp + off + 2 * GUARD
        if pinned:
            p = L.pfdHostAlloc(n)
            allocs.append(p)
            mem = np.ctypeslib.as_array((C.c_uint8 * n).from_address(p))
        else:
            mem = np.zeros(n, np.uint8)
        mem[:] = 5
        bufs.append(mem)
        ctxs.append(L.pfCreateContext(mem.ctypes.data + GUARD + off, w, h, *fmt))
    for run in range(2):
        for i, ctx in enumerate(ctxs):
            bufs[i][:] = 5
            _scene(ctx, i)
        print(f"{len(ctxs)} contexts, run {run}", flush=True)
        L.pfSubmitBatch((C.c_void_p * len(ctxs))(*ctxs), len(ctxs))
        for i, (w, h, fmt, bpp, off, pinned) in enumerate(frames):
            L.pfMakeCurrent(ctxs[i])
            assert L.pfGetError() == 0
            a = GUARD + off
            got = bufs[i][a:a + w * h * bpp]
            # Pixels a clear leaves as they were keep the first run's depths.
            if run == 0:
                assert np.array_equal(got, want[i]), f"frame {i} {frames[i]}"
            assert (bufs[i][:a] == 5).all() and (bufs[i][a + w * h * bpp:] == 5).all(), f"frame {i} {frames[i]}: past its target"
    for ctx in ctxs:
        L.pfMakeCurrent(ctx)
        L.pfDeleteContext(ctx)
    L.pfMakeCurrent(None)
    for p in allocs:
        L.pfdHostFree(p)
