"""Inputs of a frame on their way to the GPU: many array draws (more regions
than one upload launch takes, more bytes than its block), textures around
the size from which they are staged, draws from the heap (first frame) and
from the frame's page-locked block (second), and a change of render target
between draws.  Every frame must equal the oracle's."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from conftest import OracleExecutor

pytestmark = pytest.mark.gpu

W, H = 96, 64


class FB(C.Structure):
    _fields_ = [("texture", C.c_void_p), ("zbuffer", C.c_void_p)]


def _f(*v):
    return [C.c_float(float(x)) for x in v]


def _draws(L, rng, count, verts, keep):
    for k in range(count):
        n = verts + k % 7
        pos = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
        uv = rng.uniform(0, 1, (n, 2)).astype(np.float32)
        col = rng.integers(0, 256, (n, 4)).astype(np.uint8)
        idx = rng.integers(0, n, 30).astype(np.uint16 if k % 2 else np.uint32)
        keep.append((pos, uv, col, idx))
        L.pfEnable(0x100 | 0x400 | 0x800)
        L.pfVertexPointer(3, 10, 0, C.c_void_p(pos.ctypes.data))
        L.pfTexCoordPointer(10, 0, C.c_void_p(uv.ctypes.data))
        L.pfColorPointer(4, 0, 0, C.c_void_p(col.ctypes.data))
        L.pfDrawElements(2, len(idx), 1 if k % 2 else 5, C.c_void_p(idx.ctypes.data))
        pos[:] = 9                                    # the frame holds its own copies
        uv[:] = 9
        col[:] = 9
        idx[:] = 0


def _run(count, verts, tex, typ, frames=2):
    L = pf.lib()
    L.pfGenTexture.restype = C.c_void_p
    L.pfGenFramebuffer.restype = FB
    rng = np.random.default_rng(3)
    buf = np.zeros(W * H + 16, np.uint32)
    ctx = C.c_void_p(L.pfCreateContext(buf.ctypes.data, W, H, 7, 0))
    L.pfMakeCurrent(ctx)
    texels = rng.uniform(0, 1, (tex[1], tex[0], 4)).astype(np.float32) if typ == 10 else \
        rng.integers(0, 2**32, (tex[1], tex[0]), np.uint32)
    t = C.c_void_p(L.pfGenTexture(C.c_void_p(texels.ctypes.data), tex[0], tex[1], 7, typ))
    L.pfBindTexture(t)
    L.pfEnable(0x1 | 0x8)
    L.pfDisable(0x10)
    fb = L.pfGenFramebuffer(W, H, 7, 0)
    L.pfBindFramebuffer(C.byref(fb))
    keep, out = [], []
    for _ in range(frames):
        L.pfClear(3)
        _draws(L, rng, count, verts, keep)
        L.pfEnable(0x2)                               # the other target: runs the frame so far
        L.pfClear(3)
        _draws(L, rng, max(1, count // 3), verts, keep)
        L.pfDisable(0x2)
        L.pfFinish()
        L.pfEnable(0x2)
        px = np.zeros(W * H, np.uint32)
        L.pfReadPixels(0, 0, W, H, 7, 0, C.c_void_p(px.ctypes.data))
        L.pfDisable(0x2)
        out += [buf[:W * H].copy(), px]
    assert L.pfGetError() == 0
    L.pfDeleteFramebuffer(C.byref(fb))
    L.pfDeleteTexture(C.byref(t), False)
    L.pfDeleteContext(ctx)
    L.pfMakeCurrent(None)
    return out


@pytest.mark.parametrize("count,verts,tex,typ", [
    (1, 30, (5, 3), 0), (9, 40, (181, 181), 0), (60, 700, (182, 181), 0), (25, 2000, (360, 370), 0),
    (3, 12000, (64, 64), 10), (2, 30000, (400, 333), 10), (4, 30, (800, 700), 0)])
def test_uploads_match_oracle(count, verts, tex, typ):
    print(count, verts, tex, typ, flush=True)
    with OracleExecutor():
        want = _run(count, verts, tex, typ)
    pf.lib().pfxSetExecutor(None, None)
    got = _run(count, verts, tex, typ)
    for k, (a, b) in enumerate(zip(want, got)):
        assert len(np.unique(a)) > 50
        assert np.array_equal(a, b), f"image {k}: {np.count_nonzero(a != b)} pixels differ"


def _images(sizes, seed):
    L = pf.lib()
    w, h = 260, 200
    rng = np.random.default_rng(seed)
    buf = np.zeros(w * h + 16, np.uint32)
    ctx = C.c_void_p(L.pfCreateContext(buf.ctypes.data, w, h, 7, 0))
    L.pfMakeCurrent(ctx)
    L.pfDisable(0x10)
    out = []
    for _ in range(2):
        L.pfClear(3)
        for k, (iw, ih, fmt, typ, bpp) in enumerate(sizes):
            px = rng.integers(0, 256, iw * ih * bpp).astype(np.uint8)
            L.pfRasterPos3f(*_f(-1 + 0.1 * k, 1 - 0.1 * k, 0.0))
            L.pfPixelZoom(*_f(0.7, 0.7))
            L.pfDrawPixels(iw, ih, fmt, typ, C.c_void_p(px.ctypes.data))
            px[:] = 3                                 # the frame holds its own copy
        L.pfFinish()
        out.append(buf[:w * h].copy())
    assert L.pfGetError() == 0
    L.pfDeleteContext(ctx)
    L.pfMakeCurrent(None)
    return out


@pytest.mark.parametrize("sizes", [
    [(181, 181, 7, 0, 4), (182, 181, 7, 0, 4), (9, 7, 7, 0, 4)],                       # 131044, 131768 bytes
    [(3, 3, 6, 0, 3), (211, 207, 6, 0, 3), (211, 208, 6, 0, 3), (256, 256, 7, 4, 2)],  # 131031, 131664, 131072
    [(640, 480, 7, 0, 4), (333, 400, 6, 0, 3), (5, 4, 9, 3, 2), (700, 500, 4, 0, 1), (16, 16, 7, 0, 4),
     (120, 90, 6, 2, 2), (1500, 900, 8, 0, 3), (40, 40, 7, 0, 4)]],
    ids=["rgba8", "raw", "mixed"])
def test_images_around_the_gathered_size_match_oracle(sizes):
    """pfDrawPixels images on both sides of the size up to which a frame's
    images are gathered, raw and RGBA8 ones in turn."""
    print(sizes, flush=True)
    with OracleExecutor():
        want = _images(sizes, 4)
    pf.lib().pfxSetExecutor(None, None)
    got = _images(sizes, 4)
    for k, (a, b) in enumerate(zip(want, got)):
        assert len(np.unique(a)) > 50
        assert np.array_equal(a, b), f"frame {k}: {np.count_nonzero(a != b)} pixels differ"
