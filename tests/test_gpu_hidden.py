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
