"""Lines at the ends of their ranges, against the oracle: ones longer than the
16-bit slope reaches, whose steps leave their bounds, and states whose depth
function and blend mode are no enum values."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from conftest import OracleExecutor, _oracle
from frames import on_frame
from test_gpu_runs import _f, _finish, _parse, _record

pytestmark = pytest.mark.gpu


def _long_lines(target, count, width):
    """Lines from corner to corner of a 50000x60000 viewport on a target of
    its top 16 rows."""
    L = pf.lib()
    w, h = 50000, 16
    buf = np.full((w * h + 16) * 8, 7, np.uint8)
    ctx = C.c_void_p(L.pfCreateContext(buf.ctypes.data, w, h, *target))
    L.pfMakeCurrent(ctx)
    rng = np.random.default_rng(11)
    L.pfViewport(0, 0, w, 60000)
    L.pfMatrixMode(1)
    L.pfLoadIdentity()
    L.pfFrustum(*_f(-0.4, 0.4, -0.4, 0.4, 0.5, 20.0))
    L.pfMatrixMode(0)
    L.pfLoadIdentity()
    L.pfDisable(0x10)
    L.pfClear(3)
    L.pfLineWidth(*_f(width))
    L.pfBegin(1)
    for k in range(count):
        for end in (1, -1) if k % 2 else (-1, 1):
            z = -rng.uniform(1, 3)
            x, y = end * rng.uniform(0.9, 0.999), (end if k % 4 < 2 else -end) * (1.0 - rng.uniform(0, 1e-4))
            L.pfColor4ub(*rng.integers(0, 256, 4).tolist())
            L.pfVertex3f(*_f(x * 0.8 * -z, y * 0.8 * -z, z))
    L.pfEnd()
    assert L.pfGetError() == 0
    return ctx, buf


@pytest.mark.parametrize("target", [(7, 0), (7, 9)], ids=["rgba8", "rgba_half"])
@pytest.mark.parametrize("count,width", [(8, 1.0), (8, 5.0), (2100, 1.0)])
def test_long_lines_match_oracle(count, width, target):
    with OracleExecutor():
        ctx, want = _long_lines(target, count, width)
        _finish(ctx)
    pf.lib().pfxSetExecutor(None, None)
    ctx, got = _long_lines(target, count, width)
    _finish(ctx)
    drawn = np.count_nonzero(want != np.roll(want, 8))
    print(count, width, target, drawn, flush=True)
    bad = np.count_nonzero(want != got)
    assert drawn > 50 and bad == 0, f"{bad} bytes differ"


DEPTH_FUNC, BLEND_MODE, STATE_WORDS = 49, 50, 232       # PFFstate, in words


@pytest.mark.parametrize("func,mode", [(6, 7), (7, 8), (8, 9), (13, 16), (0x10000, 0x10001), (0xFFFFFFFF, 0x80000003)])
def test_states_that_are_no_enum_values_match_oracle(func, mode):
    """pfdExecuteFrame takes any value: unknown functions and modes act as the
    last ones do."""
    def run(frame):
        states = np.ctypeslib.as_array(C.cast(frame.states, C.POINTER(C.c_uint32)), (frame.numStates, STATE_WORDS))
        states[:, 48] |= 0xC                            # depth test and blending
        states[:, DEPTH_FUNC], states[:, BLEND_MODE] = func, mode
        frame.cmds[0].clearDepth = -2.0                 # the last function is "greater or equal"
        return run.execute(C.byref(frame))

    L = pf.lib()
    out = []
    for run.execute in (lambda f: _oracle.pforacle_executor(f, None), L.pfdExecuteFrame):
        ctx, buf = _record(_parse("c l60"), 9, (90, 60), (7, 0))
        with on_frame(run):
            _finish(ctx)
        out.append(buf)
    assert len(np.unique(out[0].view(np.uint32))) > 100
    bad = np.count_nonzero(out[0] != out[1])
    assert bad == 0, f"{bad} bytes differ"
