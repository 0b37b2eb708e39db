"""ctypes views of a recorded frame (include/pf_frame.h) for tests that hand
frames to the C ABI themselves, with commands changed or added that the host
library does not record."""
import ctypes as C

import pixelforge_amd as pf

CLEAR, DRAW, PIXELS, FOG, POINTS, LINES = 1, 2, 3, 4, 5, 6
PIXELS_RECT = 0x80000000


class Cmd(C.Structure):
    _fields_ = [("kind", C.c_uint32), ("first", C.c_uint32), ("last", C.c_uint32), ("clearColor", C.c_uint32),
                ("clearDepth", C.c_float), ("pad", C.c_uint32 * 3)]


class Pixels(C.Structure):
    _fields_ = [("pixels", C.c_void_p), ("width", C.c_uint32), ("height", C.c_uint32), ("source", C.c_uint32),
                ("xScreen", C.c_int32), ("yScreen", C.c_int32), ("xMin", C.c_int32), ("yMin", C.c_int32),
                ("xMax", C.c_int32), ("yMax", C.c_int32), ("zPos", C.c_float), ("invXLen", C.c_float),
                ("invYLen", C.c_float), ("flags", C.c_uint32), ("depthFunc", C.c_uint32), ("blendMode", C.c_uint32),
                ("fogMode", C.c_uint32), ("fogDensity", C.c_float), ("fogStart", C.c_float), ("fogEnd", C.c_float),
                ("fogColor", C.c_uint32)]


class Triangles(C.Structure):
    _fields_ = [("count", C.c_uint32), ("position", C.c_void_p), ("color", C.c_void_p), ("texcoord", C.c_void_p),
                ("normal", C.c_void_p), ("info", C.c_void_p), ("vertexId", C.c_void_p)]


class Frame(C.Structure):
    _fields_ = [("width", C.c_uint32), ("height", C.c_uint32), ("color", C.c_void_p), ("depth", C.c_void_p),
                ("tris", Triangles), ("states", C.c_void_p), ("numStates", C.c_uint32), ("textures", C.c_void_p),
                ("numTextures", C.c_uint32), ("cmds", C.POINTER(Cmd)), ("numCmds", C.c_uint32),
                ("pixelOps", C.POINTER(Pixels)), ("numPixelOps", C.c_uint32), ("points", C.c_void_p),
                ("numPoints", C.c_uint32), ("lines", C.c_void_p), ("numLines", C.c_uint32), ("arrays", C.c_void_p),
                ("numArrays", C.c_uint32), ("target", C.c_uint32)]


def with_commands(frame, extra):
    """A copy of `frame` with the commands `extra` after its own; it keeps
    its command array alive."""
    out = Frame.from_buffer_copy(frame)
    n = frame.numCmds
    out.keep = (Cmd * (n + len(extra)))(*[Cmd.from_buffer_copy(frame.cmds[k]) for k in range(n)], *extra)
    out.cmds = C.cast(out.keep, C.POINTER(Cmd))
    out.numCmds = n + len(extra)
    return out


class on_frame:
    """Context manager: frames of the host library go to `fn(Frame)`, whose
    result is the frame's return code (None: 0)."""

    def __init__(self, fn):
        self.error = None

        def run(frame, user):
            try:
                return fn(C.cast(frame, C.POINTER(Frame))[0]) or 0
            except BaseException as e:                            # not across the C frames
                self.error = e
                return -3
        self.cb = pf.EXECUTOR(run)

    def __enter__(self):
        pf.lib().pfxSetExecutor(C.cast(self.cb, C.c_void_p), None)
        return self

    def __exit__(self, *exc):
        pf.lib().pfxSetExecutor(None, None)
        if self.error is not None and exc[0] is None:
            raise self.error
