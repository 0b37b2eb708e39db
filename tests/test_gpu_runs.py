"""Work between triangle draws on the GPU -- runs of rects, images, fog,
points and lines, in every order -- against the oracle executing the same
recorded frame, bit for bit: runs of one operation up to several chunks of
256, operations off the target and across tile edges, narrow and wide
targets, several frames in one job, and replays of the captured graph."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from conftest import OracleExecutor

pytestmark = pytest.mark.gpu

DEPTH_TEST, BLEND = 0x8, 0x4
# (format, type) of pfDrawPixels images and bytes per texel: RGBA8 goes up as
# it is, the others are decoded.
IMAGES = [(7, 0, 4), (6, 0, 3), (7, 4, 2), (4, 10, 4), (7, 0, 4)]


def _f(*v):
    return [C.c_float(float(x)) for x in v]


def _prims(L, rng, mode, n, size=1.0):
    L.pfPointSize(*_f(size))
    L.pfLineWidth(*_f(size))
    L.pfBegin(mode)
    for _ in range(n * (1, 2, 3)[mode]):
        L.pfColor4ub(*rng.integers(0, 256, 4).tolist())
        L.pfVertex3f(*_f(*rng.uniform(-1.2, 1.2, 2), rng.uniform(-1, 1)))
    L.pfEnd()


def _rects(L, rng, n):
    for _ in range(n):
        a, e = rng.uniform(-1.3, 1.1, 2), rng.uniform(0.0, 0.5, 2)
        L.pfColor4ub(*rng.integers(0, 256, 4).tolist())
        L.pfRectf(*_f(*a, *(a + e)))


def _images(L, rng, n):
    for _ in range(n):
        fmt, typ, bpp = IMAGES[rng.integers(len(IMAGES))]
        w, h = (int(v) for v in rng.integers(1, 24, 2))
        px = rng.integers(0, 256, w * h * bpp).astype(np.uint8)
        if typ == 10:
            px = rng.uniform(0, 1, w * h).astype(np.float32)
        L.pfRasterPos3f(*_f(*rng.uniform(-1.1, 1.0, 2), rng.uniform(-1, 1)))
        L.pfPixelZoom(*_f(*rng.choice([0.5, 1.0, 2.5], 2)))
        L.pfDrawPixels(w, h, fmt, typ, C.c_void_p(px.ctypes.data))


def _fog(L, rng, n):
    for _ in range(n):
        L.pfFogi(0, int(rng.integers(0, 3)))
        s = rng.uniform(-1, 0)
        L.pfFogf(2, *_f(s))
        L.pfFogf(3, *_f(s + rng.uniform(0.1, 1.0)))
        L.pfFogfv(4, (C.c_float * 4)(*rng.uniform(0, 1, 4)))
        L.pfFogProcess()


STEPS = {"t": lambda L, r, n: _prims(L, r, 2, n), "p": lambda L, r, n: _prims(L, r, 0, n, float(r.choice([1, 3, 6.5]))),
         "l": lambda L, r, n: _prims(L, r, 1, n, float(r.choice([1, 1, 3]))), "r": _rects, "i": _images, "f": _fog,
         "c": lambda L, r, n: L.pfClear(3)}


def _record(program, seed, size, target):
    """A context with `program` recorded: a string of step letters, each
    with a count."""
    L = pf.lib()
    w, h = size
    buf = np.full((w * h + 16) * 16, 7, np.uint8)
    ctx = C.c_void_p(L.pfCreateContext(buf.ctypes.data, w, h, *target))
    assert ctx.value
    L.pfMakeCurrent(ctx)
    rng = np.random.default_rng(seed)
    L.pfDisable(0x10)
    for step, n in program:
        for bit in (DEPTH_TEST, BLEND):
            (L.pfEnable if rng.random() < 0.6 else L.pfDisable)(bit)
        L.pfBlendFunc(int(rng.integers(0, 8)))
        L.pfDepthFunc(int(rng.integers(0, 6)))
        STEPS[step](L, rng, n)
    assert L.pfGetError() == 0
    return ctx, buf


def _finish(ctx):
    L = pf.lib()
    L.pfMakeCurrent(ctx)
    L.pfFinish()
    err = L.pfGetError()
    L.pfDeleteContext(ctx)
    L.pfMakeCurrent(None)
    assert err == 0, L.pfdLastError()


def _parse(text):
    return [(w[0], int(w[1:] or 1)) for w in text.split()]


PROGRAMS = [
    "r1", "c r1 f1", "c t9 r255", "c t9 r256 i3", "c t9 r257 f1 r2", "c t9 i40 r600 i5 f2 r1",
    "c p5 l5 r5 i5 f1 t5 r5 p5 c i4 r4", "t4 f1 p9 t4 l9 r9 t4", "c c r3 c t5 p4 p4 r2", "i3 c", "p1 l1",
]


@pytest.mark.parametrize("target", [(7, 0), (6, 2), (9, 3), (7, 9), (6, 10)], ids=["rgba8", "rgb565", "bgra5551",
                                                                                   "rgba_half", "rgb_float"])
@pytest.mark.parametrize("size", [(64, 48), (37, 91), (1, 5)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_runs_match_oracle(size, target):
    for k, text in enumerate(PROGRAMS):
        print(f"{size} {target} {text}", flush=True)
        program = _parse(text)
        with OracleExecutor():
            ctx, want = _record(program, k, size, target)
            _finish(ctx)
        pf.lib().pfxSetExecutor(None, None)
        ctx, got = _record(program, k, size, target)
        _finish(ctx)
        bad = np.count_nonzero(want != got)
        assert bad == 0, f"{text} at {size}, target {target}: {bad} bytes differ"


@pytest.mark.parametrize("target", [(7, 0), (7, 9)], ids=["rgba8", "rgba_half"])
@pytest.mark.parametrize("size", [(603, 401), (16, 2000), (2000, 16), (80, 64)], ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("text", ["c p2047 l2047", "c t9 p2049 l2048 p700 l600 p1", "c p70000", "c l5000 p5000 l64"])
def test_long_runs_match_oracle(text, size, target):
    """Runs around the length from which tiles walk only the groups marked
    for them, and ones of many groups; long, steep, flat and thick lines and
    discs across tile edges."""
    for seed in (100, 101, 102):
        print(f"{size} {target} {text} {seed}", flush=True)
        program = _parse(text)
        with OracleExecutor():
            ctx, want = _record(program, seed, size, target)
            _finish(ctx)
        pf.lib().pfxSetExecutor(None, None)
        ctx, got = _record(program, seed, size, target)
        _finish(ctx)
        bad = np.count_nonzero(want != got)
        assert bad == 0, f"{text} at {size}, target {target}, seed {seed}: {bad} bytes differ"


def test_runs_of_several_frames_replayed():
    """Frames whose k-th runs differ in kind, in one job: the first run and
    two replays of its graph equal the oracle's frames."""
    L = pf.lib()
    frames = [(PROGRAMS[6], (64, 48)), (PROGRAMS[5], (130, 17)), (PROGRAMS[7], (33, 33)), ("c t6", (40, 40)), ("c l9 i2", (50, 20)),
              ("c p3000 l3000", (300, 200)), ("c r4 p2500", (400, 300))]
    want = []
    with OracleExecutor():
        for k, (text, size) in enumerate(frames):
            ctx, buf = _record(_parse(text), 50 + k, size, (7, 0))
            _finish(ctx)
            want.append(buf)
    recs = [_record(_parse(text), 50 + k, size, (7, 0)) for k, (text, size) in enumerate(frames)]
    ctxs = [c for c, _ in recs]
    L.pfxSetBatchExecutor(C.cast(L.pfdCaptureBatchExecutor, C.c_void_p), None)
    try:
        L.pfSubmitBatch((C.c_void_p * len(ctxs))(*[c.value for c in ctxs]), len(ctxs))
    finally:
        L.pfxSetBatchExecutor(None, None)
    job = L.pfdTakeCapturedJob()
    assert job
    cap = pf.Captured(job, [], [], [])
    try:
        snap = cap.snapshot()
        for run in range(3):
            cap.restore(snap)
            assert L.pfdJobLaunch(cap.job) == 0 and L.pfdJobSync(cap.job) == 0 and L.pfdJobDownload(cap.job) == 0
            for k, (_, got) in enumerate(recs):
                assert np.array_equal(got, want[k]), f"run {run}, frame {k}"
    finally:
        cap.close()
        for c in ctxs:
            L.pfMakeCurrent(c)
            L.pfDeleteContext(c)
        L.pfMakeCurrent(None)
