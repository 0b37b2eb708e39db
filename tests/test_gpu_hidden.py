"""Records the raster kernel drops as hidden behind a block's pixels: frames
of many layers, whose depth functions change within a tile's list so that
pixels' depths move both ways, must equal the oracle bit for bit, and the
covered samples must be counted as if nothing were dropped, at every tile
size and raster mode."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from conftest import OracleExecutor

pytestmark = pytest.mark.gpu

LESS, LEQUAL, GREATER, GEQUAL = 2, 3, 4, 5


def _f(*v):
    return [C.c_float(float(x)) for x in v]


def _record(seed, size, target, funcs, test_off, three_d, tris=4000, run=25):
    """Triangles from a few pixels to the whole frame, drawn in runs of `run`
    with one of `funcs`, a share `test_off` of the runs without a depth test;
    a third of the runs blended; z spread, constant, and exactly 0 or tiny."""
    L = pf.lib()
    w, h = size
    buf = np.full((w * h + 16) * 16, 9, np.uint8)
    ctx = C.c_void_p(L.pfCreateContext(buf.ctypes.data, w, h, *target))
    L.pfMakeCurrent(ctx)
    rng = np.random.default_rng(seed)
    L.pfDisable(0x10)
    L.pfClearDepth(*_f(rng.choice([1.0, 0.0, -3.0]) if max(funcs) >= GREATER else 3.4028234663852886e38))
    L.pfClear(3)
    if three_d:
        L.pfMatrixMode(1)
        L.pfLoadIdentity()
        L.pfFrustum(*_f(-0.4, 0.4, -0.4, 0.4, 0.5, 20.0))
        L.pfMatrixMode(0)
        L.pfLoadIdentity()
    for _ in range(tris // run):
        (L.pfDisable if rng.random() < test_off else L.pfEnable)(0x8)
        L.pfDepthFunc(int(rng.choice(funcs)))
        (L.pfEnable if rng.random() < 0.33 else L.pfDisable)(0x4)
        L.pfBlendFunc(int(rng.integers(0, 8)))
        size_k, z_k = rng.choice([0.05, 0.4, 2.0]), rng.integers(0, 4)
        L.pfBegin(2)
        for _ in range(run):
            c, z0 = rng.uniform(-1, 1, 2), rng.uniform(-0.9, 0.9)
            for _ in range(3):
                x, y = c + size_k * rng.uniform(-1, 1, 2)
                z = (rng.uniform(-0.9, 0.9), z0, z0 + rng.uniform(-1e-3, 1e-3), rng.choice([0.0, 1e-38, -1e-35, 0.5]))[z_k]
                if three_d:
                    z = -3.0 + 2.0 * z
                    x, y = -x * z, -y * z
                L.pfColor4ub(*rng.integers(0, 256, 4).tolist())
                L.pfVertex3f(*_f(x, y, z))
        L.pfEnd()
    assert L.pfGetError() == 0
    return ctx, buf


CASES = {
    "less": dict(funcs=[LESS], test_off=0.0, three_d=False),
    "less_equal_3d": dict(funcs=[LESS, LEQUAL], test_off=0.0, three_d=True),
    "greater": dict(funcs=[GREATER, GEQUAL], test_off=0.0, three_d=False),
    "greater_3d": dict(funcs=[GREATER], test_off=0.0, three_d=True),
    "all": dict(funcs=[0, 1, 2, 3, 4, 5], test_off=0.05, three_d=False),
    "mostly_less": dict(funcs=[2] * 12 + [3] * 6 + [0, 4], test_off=0.01, three_d=False),
    "less_and_equal_3d": dict(funcs=[0, 1, 2, 3], test_off=0.0, three_d=True),
}


@pytest.mark.parametrize("target", [(7, 0), (6, 2), (7, 9)], ids=["rgba8", "rgb565", "rgba_half"])
@pytest.mark.parametrize("name", CASES)
def test_layers_match_oracle(name, target):
    L = pf.lib()
    size = (101, 75)
    with OracleExecutor() as ex:
        ctx, want = _record(5, size, target, **CASES[name])
        L.pfFinish()
        samples = ex.fragments
        L.pfDeleteContext(ctx)
    ctx, got = _record(5, size, target, **CASES[name])
    L.pfxSetExecutor(C.cast(L.pfdCaptureExecutor, C.c_void_p), None)
    try:
        L.pfFinish()
    finally:
        L.pfxSetExecutor(None, None)
    cap = pf.Captured(L.pfdTakeCapturedJob(), [], [], [])
    try:
        depth = cap.targets()[0][1]
        snap = got.copy(), depth.copy()
        for shift, mode in [(3, 0), (3, 1), (4, 2), (4, 0), (4, 1), (5, 0), (5, 1), (6, 0), (6, 1)]:
            print(f"{name} {target} tile {1 << shift} mode {mode}", flush=True)
            cfg = pf.PFDconfig()
            cfg.tileShift, cfg.rasterMode = shift, mode
            assert L.pfdJobSetConfig(cap.job, C.byref(cfg)) == 0
            for run in range(2):                                  # sizing run, graph
                got[:], depth[:] = snap
                assert L.pfdJobUploadTargets(cap.job) == 0
                assert L.pfdJobLaunch(cap.job) == 0 and L.pfdJobSync(cap.job) == 0 and L.pfdJobDownload(cap.job) == 0
                bad = np.count_nonzero(got != want)
                assert bad == 0, f"{name} tile {1 << shift} mode {mode} run {run}: {bad} bytes differ"
                st = pf.PFDstats()
                assert L.pfdJobStats(cap.job, C.byref(st)) == 0
                assert int(st.fragments) == samples
    finally:
        cap.close()
        L.pfMakeCurrent(ctx)
        L.pfDeleteContext(ctx)
        L.pfMakeCurrent(None)


def _jobs_match_oracle(record, size, what):
    """`record`: makes a context with a recorded frame, and its buffer.  The
    frame at every tile size and raster mode, a sizing run and a replay each,
    against the oracle's."""
    L = pf.lib()
    with OracleExecutor() as ex:
        ctx, want = record()
        L.pfFinish()
        samples = ex.fragments
        L.pfDeleteContext(ctx)
    ctx, got = record()
    L.pfxSetExecutor(C.cast(L.pfdCaptureExecutor, C.c_void_p), None)
    try:
        L.pfFinish()
    finally:
        L.pfxSetExecutor(None, None)
    cap = pf.Captured(L.pfdTakeCapturedJob(), [], [], [])
    try:
        depth = cap.targets()[0][1]
        snap = got.copy(), depth.copy()
        for shift, mode in [(3, 0), (3, 1), (4, 2), (4, 0), (4, 1), (5, 0), (5, 1), (6, 0), (6, 1)]:
            print(f"{what} tile {1 << shift} mode {mode}", flush=True)
            cfg = pf.PFDconfig()
            cfg.tileShift, cfg.rasterMode = shift, mode
            assert L.pfdJobSetConfig(cap.job, C.byref(cfg)) == 0
            for run in range(2):
                got[:], depth[:] = snap
                assert L.pfdJobUploadTargets(cap.job) == 0
                assert L.pfdJobLaunch(cap.job) == 0 and L.pfdJobSync(cap.job) == 0 and L.pfdJobDownload(cap.job) == 0
                bad = np.count_nonzero(got != want)
                assert bad == 0, f"{what} tile {1 << shift} mode {mode} run {run}: {bad} bytes differ"
                st = pf.PFDstats()
                assert L.pfdJobStats(cap.job, C.byref(st)) == 0
                assert int(st.fragments) == samples
    finally:
        cap.close()
        L.pfMakeCurrent(ctx)
        L.pfDeleteContext(ctx)
        L.pfMakeCurrent(None)


def _record_lit(seed, size, target, model, textured):
    """Layers of lit triangles, back to front and front to back, a third of
    the runs blended, some without lighting."""
    L = pf.lib()
    L.pfGenTexture.restype = C.c_void_p
    w, h = size
    buf = np.full((w * h + 16) * 8, 9, np.uint8)
    ctx = C.c_void_p(L.pfCreateContext(buf.ctypes.data, w, h, *target))
    L.pfMakeCurrent(ctx)
    rng = np.random.default_rng(seed)
    L.pfDisable(0x10)
    L.pfEnable(0x8)
    L.pfClear(3)
    L.pfMatrixMode(1)
    L.pfLoadIdentity()
    L.pfFrustum(*_f(-0.4, 0.4, -0.4, 0.4, 0.5, 20.0))
    L.pfMatrixMode(0)
    L.pfLoadIdentity()
    L.pfLightModel(model)
    for k in range(3):
        L.pfLightfv(k, 7, (C.c_float * 3)(*rng.uniform(-2, 2, 3)))
        L.pfLightfv(k, 3, (C.c_float * 3)(*rng.uniform(0.2, 0.7, 3)))
        L.pfLightfv(k, 4, (C.c_float * 3)(*rng.uniform(0.1, 0.5, 3)))
        L.pfEnableLight(k)
    L.pfMaterialfv(2, 4, (C.c_float * 3)(0.8, 0.7, 0.9))
    L.pfMaterialf(2, 6, C.c_float(16.0))
    if textured:
        texels = rng.integers(0, 2**32, (17, 33), np.uint32)
        tex = C.c_void_p(L.pfGenTexture(C.c_void_p(texels.ctypes.data), 33, 17, 7, 0))
        L.pfTextureParameter(tex, pf.PF_REPEAT, pf.PF_BILINEAR)
        L.pfBindTexture(tex)
        KEEP.append(texels)
    for _ in range(120):
        (L.pfEnable if textured and rng.random() < 0.8 else L.pfDisable)(0x1)
        (L.pfEnable if rng.random() < 0.8 else L.pfDisable)(0x40)
        (L.pfEnable if rng.random() < 0.33 else L.pfDisable)(0x4)
        L.pfBlendFunc(int(rng.integers(0, 8)))
        L.pfDepthFunc(int(rng.choice([LESS, LESS, LESS, LEQUAL, 0])))
        size_k, far = rng.choice([0.1, 0.5, 2.0]), rng.uniform(-0.9, 0.9)
        L.pfBegin(2)
        for _ in range(20):
            c = rng.uniform(-1, 1, 2)
            for _ in range(3):
                z = -3.0 + 2.0 * (far + rng.uniform(-0.05, 0.05))
                x, y = c + size_k * rng.uniform(-1, 1, 2)
                L.pfColor4ub(*rng.integers(0, 256, 4).tolist())
                L.pfNormal3f(*_f(*rng.normal(0, 1, 3)))
                L.pfTexCoord2f(*_f(*rng.uniform(-2, 3, 2)))
                L.pfVertex3f(*_f(-x * z, -y * z, z))
        L.pfEnd()
    assert L.pfGetError() == 0
    return ctx, buf


KEEP = []                                                         # texels of recorded frames


@pytest.mark.parametrize("target", [(7, 0), (7, 9)], ids=["rgba8", "rgba_half"])
@pytest.mark.parametrize("model,textured", [(1, False), (1, True), (0, True)], ids=["phong", "phong_tex", "gouraud_tex"])
def test_lit_and_textured_layers_match_oracle(model, textured, target):
    size = (101, 75)
    _jobs_match_oracle(lambda: _record_lit(7, size, target, model, textured), size, f"model {model} {textured} {target}")


def _weights(corners, w, h):
    """Edge values of a triangle of screen corners at pixel (0, 0), its
    largest magnitude of one within 128 pixels of the target, and their sum."""
    (x1, y1), (x2, y2), (x3, y3) = [(int(x), int(y)) for x, y in corners]
    a = (y3 - y2, y1 - y3, y2 - y1)
    b = (x2 - x3, x3 - x1, x1 - x2)
    c = [-(ox * a[k] + oy * b[k]) for k, (ox, oy) in enumerate(((x2, y2), (x3, y3), (x1, y1)))]
    far = max(abs(a[k] * x + b[k] * y + c[k]) for k in range(3) for x in (-128, w + 128) for y in (-128, h + 128))
    return c, far, sum(c)


def _record_wrapping(seed, size, func):
    """Seventy layers, then triangles around the target so large that the sum
    of a pixel's three weights leaves 32 bits where no weight does: their
    barycentric coordinates do not add up to one."""
    L = pf.lib()
    w, h = size
    buf = np.full((w * h + 16) * 4, 9, np.uint8)
    ctx = C.c_void_p(L.pfCreateContext(buf.ctypes.data, w, h, 7, 0))
    L.pfMakeCurrent(ctx)
    rng = np.random.default_rng(seed)
    sign = -1.0 if func >= GREATER else 1.0
    for matrix in (1, 0):
        L.pfMatrixMode(matrix)
        L.pfLoadIdentity()
    L.pfDisable(0x10)
    L.pfEnable(0x8)
    L.pfClearDepth(*_f(sign * 3e38))
    L.pfClear(3)
    L.pfDepthFunc(func)

    def triangle(corners, z):
        L.pfBegin(2)
        L.pfColor4ub(*rng.integers(0, 256, 4).tolist())
        for (x, y), zk in zip(corners, z):
            # Half a pixel off the edge of the truncation to whole pixels.
            L.pfVertex3f(*_f(2.0 * (x + 0.5 * np.sign(x)) / (w - 1) - 1.0, 1.0 - 2.0 * (y + 0.5 * np.sign(y)) / (h - 1), zk))
        L.pfEnd()

    for k in range(70):
        d = sign * (1.0 + (70 - k) * 0.01)                        # the layers end at a depth of 1.01
        triangle([(-9, -9), (-9, 9 * h), (9 * w, -9)], [1.0 / d] * 3)
    wrapped = 0
    for _ in range(40):
        s = rng.uniform(22000, 27000)
        corners = [(-s, -s), (-s, 2 * s), (2 * s, -s)] + rng.uniform(-0.02, 0.02, (3, 2)) * s
        if rng.random() < 0.5:
            corners = corners[[0, 2, 1]]
        corners = np.trunc(corners)
        _, far, total = _weights(corners, w, h)
        wrapped += far < 2**31 - 2**24 and abs(total) > 2**31 + 2**24
        # Behind the layers if the coordinates added up to one.
        z = sign * rng.uniform(0.3, 0.75) * (1.0 if rng.random() < 0.3 else rng.uniform(0.8, 1.25, 3)) * np.ones(3)
        triangle(corners, z)
    assert wrapped >= 20
    assert L.pfGetError() == 0
    return ctx, buf


@pytest.mark.parametrize("func", [LESS, LEQUAL, GREATER, GEQUAL])
def test_triangles_whose_weights_wrap_match_oracle(func):
    for seed, size in ((1, (101, 75)), (2, (33, 140))):
        _jobs_match_oracle(lambda: _record_wrapping(seed, size, func), size, f"function {func} size {size}")
