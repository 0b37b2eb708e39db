"""Runs of points and lines so long, on targets so large, that their marks do
not fit at one bit per group of 64: groups of 128 to 512 primitives, and none
where even that is too much; against the oracle, bit for bit.  Ends of groups
and words that are not full, primitives across tile edges and off the target,
and a narrow target of ragged sides."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from conftest import OracleExecutor
from test_gpu_runs import _f, _finish

pytestmark = pytest.mark.gpu

# Words of marks a job may have (RUN_MARK_WORDS), and primitives per word.
WORDS, PER_WORD = 16 << 20, 2048


def _shift(runs, tiles):
    """Groups of 64 << shift that the runs' marks need; 17: none fits."""
    for shift in range(17):
        if sum(tiles * -(--(-n // PER_WORD) >> shift) for n in runs) <= WORDS:
            return shift
    return 17


def _render(kind, runs, size, seed):
    L = pf.lib()
    w, h = size
    rng = np.random.default_rng(seed)
    buf = np.zeros(w * h + 16, np.uint32)
    ctx = C.c_void_p(L.pfCreateContext(buf.ctypes.data, w, h, 7, 0))
    L.pfMakeCurrent(ctx)
    L.pfDisable(0x10)
    L.pfEnable(0x8 | 0x4)
    L.pfBlendFunc(1)
    L.pfClear(3)
    L.pfPointSize(*_f(2.5))
    for k, n in enumerate(runs):
        if kind == "points":
            pos = rng.uniform(-1.02, 1.02, (n, 3)).astype(np.float32)
        else:
            a = rng.uniform(-1.0, 1.0, (n, 3))
            b = a + rng.uniform(-1, 1, (n, 3)) * [40.0 / w, 40.0 / h, 0.2]
            pos = np.stack([a, b], 1).reshape(-1, 3).astype(np.float32)
        col = rng.integers(0, 256, (len(pos), 4)).astype(np.uint8)
        L.pfEnable(0x100 | 0x400)
        L.pfVertexPointer(3, 10, 0, C.c_void_p(pos.ctypes.data))
        L.pfColorPointer(4, 0, 0, C.c_void_p(col.ctypes.data))
        L.pfDrawArrays(0 if kind == "points" else 1, 0, len(pos))
        if len(runs) > 1:
            L.pfRectf(*_f(-0.5, -0.5, -0.499, -0.499))           # ends the run
    assert L.pfGetError() == 0
    _finish(ctx)
    return buf


@pytest.mark.parametrize("kind,runs,size,shift", [
    ("points", [600001], (4096, 4096), 1),
    ("points", [524289 + 524288], (4096, 4096), 2),
    ("points", [2400000], (4095, 4081), 3),
    ("points", [3000, 700000, 64, 5000], (4096, 4090), 1),
    ("points", [513] * 260, (4096, 4096), 17),
    ("lines", [300000, 300001], (4096, 4096), 1),
    ("lines", [2049] * 257, (4096, 4095), 17),
    ("points", [6001, 70001], (37, 2311), 0),
    ("lines", [6001, 50000], (2311, 37), 0)], ids=lambda v: None if isinstance(v, list) else str(v))
def test_coarse_marks_match_oracle(kind, runs, size, shift):
    tiles = -(-size[0] // 16) * -(-size[1] // 16)
    assert _shift([n for n in runs if n >= 512], tiles) == shift
    print(kind, len(runs), size, shift, flush=True)
    with OracleExecutor():
        want = _render(kind, runs, size, 5)
    pf.lib().pfxSetExecutor(None, None)
    got = _render(kind, runs, size, 5)
    assert len(np.unique(want)) > 1000
    bad = np.count_nonzero(want != got)
    assert bad == 0, f"{bad} pixels differ"
