"""Images and parameters in page-locked memory, which the shading kernels
and one upload launch reach directly, against ordinary memory: the image is
the same bit for bit, the gradients up to the order of their final 32-bit
adds (at most 64 blocks share a texel here: 64 x 2^-24 < 1e-5 of the
largest).  Page-locked pointers are taken at 16-byte alignment and 4 bytes
past it (which goes through the job's own copy); the floats around the image
stay as they were."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from pixelforge_amd.diffmesh import DiffGrads, Scene, params_of

pytestmark = pytest.mark.gpu


def _pinned(allocs, shape, off, fill=None):
    L = pf.lib()
    L.pfdHostAlloc.restype = C.c_void_p
    L.pfdHostAlloc.argtypes = [C.c_size_t]
    L.pfdHostFree.argtypes = [C.c_void_p]
    n = int(np.prod(shape))
    at = L.pfdHostAlloc((n + 16) * 4)
    assert at
    allocs.append(at)
    whole = np.ctypeslib.as_array((C.c_float * (n + 16)).from_address(at))
    whole[:] = -7.0
    view = whole[off:off + n].reshape(shape)
    if fill is not None:
        view[...] = fill
    return whole, view


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("width,height,tex", [(1, 1, 4), (37, 29, 16), (128, 64, 128)])
def test_page_locked_equals_ordinary(width, height, tex, off):
    L = pf.lib()
    if L.pfdInit() != 0:
        pytest.fail("no GPU: " + L.pfdLastError().decode())
    allocs = []
    s = Scene(width=width, height=height, nx=12, nz=9, tex=(tex, tex), seed=31)
    try:
        s.record()
        p = [a.astype(np.float32) for a in params_of(s)]
        img = s.gpu_forward(*p)
        d = np.random.default_rng(8).normal(0, 0.1, img.shape).astype(np.float32)
        want = s.gpu_backward(*p, d)
        params, keep = s.gpu_params(*p)
        whole, texels = _pinned(allocs, p[0].shape, off, p[0])
        params.texels = texels.ctypes.data
        iw, image = _pinned(allocs, img.shape, off)
        dw, dimg = _pinned(allocs, img.shape, off, d)
        L.pfDiffRender(C.byref(params), C.c_void_p(image.ctypes.data))
        assert L.pfGetError() == 0
        assert np.array_equal(image.view(np.uint32), img.view(np.uint32))
        assert (iw[:off] == -7.0).all() and (iw[off + img.size:] == -7.0).all()
        outs = [_pinned(allocs, w.shape, off)[1] for w in want]
        g = DiffGrads(*[o.ctypes.data for o in outs])
        L.pfDiffBackward(C.byref(params), C.c_void_p(dimg.ctypes.data), C.byref(g))
        assert L.pfGetError() == 0
        for a, b in zip(outs, want):
            assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max()
    finally:
        s.close()
        for at in allocs:
            L.pfdHostFree(at)
