"""pfdJobStats of frames whose passes hold no triangles: points, lines, rects,
images and fog alone have no tile lists, whatever the device memory held
before and whatever passes came before."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from frames import DRAW, Cmd, on_frame, with_commands
from test_gpu_runs import _parse, _record

pytestmark = pytest.mark.gpu


def _stats(frame, shift):
    L = pf.lib()
    cfg = pf.PFDconfig()
    cfg.tileShift = shift
    job = C.c_void_p()
    assert L.pfdJobCreate(C.byref(frame), 1, C.byref(cfg), C.byref(job)) == 0, L.pfdLastError()
    try:
        for _ in range(2):                                        # sizing run, graph
            assert L.pfdJobUploadTargets(job) == 0 and L.pfdJobLaunch(job) == 0 and L.pfdJobSync(job) == 0
        st = pf.PFDstats()
        assert L.pfdJobStats(job, C.byref(st)) == 0
        return st
    finally:
        L.pfdJobDestroy(job)


# Program, and the commands added behind it; whether its last pass draws.
CASES = [("p9", [], False), ("l9", [], False), ("r3", [], False), ("i2 f1", [], False), ("c r3", [], False), ("c", [], False),
         ("c t30 r2", [Cmd(DRAW, 0, 0)], False), ("t30 p4", [Cmd(DRAW, 30, 30)], False), ("c t30", [], True),
         ("p3 t30 l3", [], True)]


@pytest.mark.parametrize("shift", [3, 5])
@pytest.mark.parametrize("program,extra,draws", CASES, ids=lambda v: v.replace(" ", "_") if isinstance(v, str) else None)
def test_tile_lists_are_of_the_last_pass(program, extra, draws, shift):
    L = pf.lib()
    for text in ("c t60", program):                               # the first leaves tile lists in freed device memory
        seen = []
        ctx, _ = _record(_parse(text), 3, (130, 70), (7, 0))
        with on_frame(lambda f: seen.append(_stats(with_commands(f, extra if text == program else []), shift))):
            L.pfFinish()
        L.pfDeleteContext(ctx)
        L.pfMakeCurrent(None)
        st = seen[0]
    print(program, st.busyTiles, st.maxTileList, flush=True)
    assert (st.busyTiles > 0) == draws and (st.maxTileList > 0) == draws
    assert st.busyTiles <= st.numTiles and st.maxTileList <= st.rasterTriangles
