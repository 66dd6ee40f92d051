"""Stream captures made straight through the HIP runtime that torch loaded: a
call that fails inside one ends the test, not the process."""
import ctypes

VP = ctypes.c_void_p
THREAD_LOCAL, GLOBAL, RELAXED = 1, 0, 2


def runtime():
    path = [line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line][0]
    return ctypes.CDLL(path)


class Graph:
    """The calls that `fn(stream)` makes, captured on a stream of its own."""

    def __init__(self, fn, mode=THREAD_LOCAL):
        self.hip, self.stream, self.exe = runtime(), VP(), VP()
        graph = VP()
        self._ok(self.hip.hipStreamCreateWithFlags(ctypes.byref(self.stream), 1))
        self._ok(self.hip.hipStreamBeginCapture(self.stream, mode))
        try:
            fn(self.stream.value)
        finally:
            rc = self.hip.hipStreamEndCapture(self.stream, ctypes.byref(graph))
            self.hip.hipGetLastError()
        self._ok(rc)
        n = ctypes.c_size_t()
        self._ok(self.hip.hipGraphGetNodes(graph, None, ctypes.byref(n)))
        self.nodes = n.value
        self._ok(self.hip.hipGraphInstantiate(ctypes.byref(self.exe), graph, None, None,
                                              ctypes.c_size_t(0)))
        self._ok(self.hip.hipGraphDestroy(graph))

    @staticmethod
    def _ok(rc):
        assert rc == 0, f"HIP error {rc}"

    def replay(self, stream=None):
        self._ok(self.hip.hipGraphLaunch(self.exe, VP(stream) if stream else self.stream))

    def wait(self):
        self._ok(self.hip.hipStreamSynchronize(self.stream))

    def close(self):
        if self.exe:
            self.wait()
            self._ok(self.hip.hipGraphExecDestroy(self.exe))
            self._ok(self.hip.hipStreamDestroy(self.stream))
            self.exe = VP()
