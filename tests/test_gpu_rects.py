"""Images with the rect flag that a caller of the C ABI hands over itself:
tested, blended, of several texels or another source than RGBA8.  They are
images that write no depth, as the oracle draws them; plain rects in the same
run."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from conftest import _oracle
from frames import PIXELS_RECT, Frame, Pixels, on_frame
from test_gpu_runs import _parse, _record

pytestmark = pytest.mark.gpu

DEPTH_TEST, BLEND = 0x8, 0x4
# width, height, PFF_SOURCE(format, type), bytes per texel, flags beside the rect's.
IMAGES = {
    "blended": (1, 1, 7, 4, BLEND),
    "tested": (1, 1, 7, 4, DEPTH_TEST),
    "tested_blended": (1, 1, 7, 4, DEPTH_TEST | BLEND),
    "texels": (3, 2, 7, 4, 0),
    "rgb": (1, 1, 6, 3, 0),
    "red_blended": (1, 1, 0, 1, BLEND),
    "rgba4444": (2, 2, 7 | 4 << 8, 2, DEPTH_TEST),
}


@pytest.mark.parametrize("target", [(7, 0), (6, 2), (7, 9)], ids=["rgba8", "rgb565", "rgba_half"])
@pytest.mark.parametrize("name", IMAGES)
def test_rect_images_match_oracle(name, target):
    L = pf.lib()
    w, h, source, bpp, flags = IMAGES[name]
    rng = np.random.default_rng(8)

    def run(frame):
        ops = (Pixels * frame.numPixelOps)(*[Pixels.from_buffer_copy(frame.pixelOps[k]) for k in range(frame.numPixelOps)])
        keep = []
        for k, op in enumerate(ops):
            if k % 3 == 0:
                continue                                          # stays a plain rect
            px = rng.integers(1, 256, w * h * bpp).astype(np.uint8)
            keep.append(px)
            op.pixels, op.width, op.height, op.source = px.ctypes.data, w, h, source
            op.flags = PIXELS_RECT | flags
            op.depthFunc, op.blendMode = int(rng.integers(0, 6)), int(rng.integers(0, 8))
            op.zPos = float(rng.uniform(-1, 1))
            op.invXLen, op.invYLen = 1.0 / max(1, op.xMax - op.xMin), 1.0 / max(1, op.yMax - op.yMin)
        f = Frame.from_buffer_copy(frame)
        f.pixelOps = C.cast(ops, C.POINTER(Pixels))
        n = f.width * f.height
        size = {(7, 0): 4, (6, 2): 2, (7, 9): 8}[target] * n
        color = np.ctypeslib.as_array(C.cast(f.color, C.POINTER(C.c_uint8)), (size,))
        depth = np.ctypeslib.as_array(C.cast(f.depth, C.POINTER(C.c_uint32)), (n,))
        before = color.copy(), depth.copy()
        assert _oracle.pforacle_executor(C.byref(f), None) == 0
        want = color.copy(), depth.copy()
        color[:], depth[:] = before
        assert L.pfdExecuteFrame(C.byref(f)) == 0, L.pfdLastError()
        assert np.array_equal(color, want[0]), f"{np.count_nonzero(color != want[0])} colour bytes differ"
        assert np.array_equal(depth, want[1]), f"{np.count_nonzero(depth != want[1])} depths differ"
        assert np.count_nonzero(color != before[0]) > n // 2

    print(name, target, flush=True)
    ctx, _ = _record(_parse("c t9 r24"), 6, (75, 50), target)
    with on_frame(run):
        L.pfFinish()
    L.pfDeleteContext(ctx)
    L.pfMakeCurrent(None)
