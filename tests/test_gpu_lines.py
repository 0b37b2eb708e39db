"""Lines at the ends of their ranges, against the oracle: states whose depth
function and blend mode are no enum values."""
import ctypes as C

import numpy as np
import pytest

import pixelforge_amd as pf
from conftest import _oracle
from frames import on_frame
from test_gpu_runs import _finish, _parse, _record

pytestmark = pytest.mark.gpu


DEPTH_FUNC, BLEND_MODE, STATE_WORDS = 49, 50, 232       # PFFstate, in words


@pytest.mark.parametrize("func,mode", [(6, 7), (7, 8), (8, 9), (13, 16), (0x10000, 0x10001), (0xFFFFFFFF, 0x80000003)])
def test_states_that_are_no_enum_values_match_oracle(func, mode):
    """pfdExecuteFrame takes any value: unknown functions and modes act as the
    last ones do."""
    def run(frame):
        states = np.ctypeslib.as_array(C.cast(frame.states, C.POINTER(C.c_uint32)), (frame.numStates, STATE_WORDS))
        states[:, 48] |= 0xC                            # depth test and blending
        states[:, DEPTH_FUNC], states[:, BLEND_MODE] = func, mode
        return run.execute(C.byref(frame))

    L = pf.lib()
    out = []
    for run.execute in (lambda f: _oracle.pforacle_executor(f, None), L.pfdExecuteFrame):
        ctx, buf = _record(_parse("c l60"), 9, (90, 60), (7, 0))
        with on_frame(run):
            _finish(ctx)
        out.append(buf)
    assert np.count_nonzero(out[0] != 7) > 90 * 60
    bad = np.count_nonzero(out[0] != out[1])
    assert bad == 0, f"{bad} bytes differ"
