"""HIP graphs of the C ABI's calls, for the GPU tests."""
import ctypes


class Capture:
    """HIP stream capture through the library's own runtime: mode 0 global, 2 relaxed."""

    def __init__(self, ctx, stream, mode):
        self.lib, self.stream, self.graph, self.exec = ctx.lib, ctypes.c_void_p(stream), ctypes.c_void_p(), ctypes.c_void_p()
        self.mode = mode

    def __enter__(self):
        assert self.lib.hipStreamBeginCapture(self.stream, self.mode) == 0
        return self

    def __exit__(self, *exc):
        assert self.lib.hipStreamEndCapture(self.stream, ctypes.byref(self.graph)) == 0
        if exc[0] is None and self.graph:
            assert self.lib.hipGraphInstantiate(ctypes.byref(self.exec), self.graph, None, None, ctypes.c_size_t(0)) == 0

    def launch(self):
        assert self.lib.hipGraphLaunch(self.exec, self.stream) == 0

    def close(self):
        for f, h in ((self.lib.hipGraphExecDestroy, self.exec), (self.lib.hipGraphDestroy, self.graph)):
            if h:
                assert f(h) == 0
