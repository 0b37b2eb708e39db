"""A differentiable frame without a clear whose triangles leave whole tiles
alone: those pixels take the target's colour and have no part in the
gradients, as in the same frame with a clear to that colour, whatever the
job's memory held before."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from frames import CLEAR, DRAW, Cmd, Frame, on_frame
from pixelforge_amd.diffmesh import DiffGrads, Scene

pytestmark = pytest.mark.gpu


class Params(C.Structure):              # PFDdiffParams
    _fields_ = [("texture", C.c_int32), ("texels", C.c_void_p), ("numVertices", C.c_uint32),
                ("vertexColors", C.c_void_p), ("lightDiffuse", C.c_void_p), ("lightSpecular", C.c_void_p)]


def _run(s, frame, tris, clear, dimg):
    """Image and gradients of the first `tris` triangles."""
    L = pf.lib()
    f = Frame.from_buffer_copy(frame)
    own = frame.cmds[0]
    assert own.kind == CLEAR and frame.numCmds == 2
    cmds = (Cmd * 2)(Cmd.from_buffer_copy(own), Cmd(DRAW, 0, tris))
    n = f.width * f.height
    color = np.ctypeslib.as_array(C.cast(f.color, C.POINTER(C.c_uint32)), (n,))
    depth = np.ctypeslib.as_array(C.cast(f.depth, C.POINTER(C.c_float)), (n,))
    color[:], depth[:] = own.clearColor, own.clearDepth
    f.cmds = C.cast(C.byref(cmds, 0 if clear else C.sizeof(Cmd)), C.POINTER(Cmd))
    f.numCmds = 2 if clear else 1
    job = C.c_void_p()
    assert L.pfdDiffCreate(C.byref(f), C.byref(job)) == 0, L.pfdLastError()
    try:
        p = Params(0, s.texels.ctypes.data, s.nv, s.colors.ctypes.data, s.ldiff.ctypes.data, s.lspec.ctypes.data)
        img = np.zeros((s.H, s.W, 4), np.float32)
        assert L.pfdDiffForward(job, C.byref(p), img.ctypes.data_as(C.c_void_p)) == 0, L.pfdLastError()
        g = [np.zeros_like(s.texels), np.zeros_like(s.colors), np.zeros((8, 3), np.float32), np.zeros((8, 3), np.float32)]
        grads = DiffGrads(*[a.ctypes.data for a in g])
        assert L.pfdDiffBackward(job, C.byref(p), dimg.ctypes.data_as(C.c_void_p), C.byref(grads)) == 0, L.pfdLastError()
        return img, g
    finally:
        L.pfdJobDestroy(job)


@pytest.mark.parametrize("tris", [0, 420, 900])
def test_tiles_left_alone_take_the_target(tris):
    L = pf.lib()
    L.pfdDiffCreate.argtypes = [C.c_void_p, C.c_void_p]
    if L.pfdInit() != 0:
        pytest.fail("no GPU: " + L.pfdLastError().decode())
    s = Scene(width=150, height=110, nx=30, nz=30, tex=(16, 16), lights=2, seed=31)
    dimg = np.random.default_rng(31).normal(0, 1, (s.H, s.W, 4)).astype(np.float32)
    out = {}

    def run(frame):
        _run(s, frame, frame.tris.count, True, dimg)              # winners of every pixel in freed memory
        out["clear"] = _run(s, frame, tris, True, dimg)
        _run(s, frame, frame.tris.count, True, dimg)
        out["none"] = _run(s, frame, tris, False, dimg)

    try:
        s.record()
        with on_frame(run):
            L.pfFinish()
    finally:
        s.close()
    (img, g), (want, gw) = out["none"], out["clear"]
    print(tris, np.count_nonzero(np.abs(want - want[0, 0]).max(-1) > 0), flush=True)
    assert np.array_equal(img, want)
    for name, a, b in zip(("texels", "colors", "ldiff", "lspec"), g, gw):
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b), name
        assert np.any(b) == (tris > 0), name
