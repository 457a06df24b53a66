"""A GpuContext whose library calls are logged instead of run, for tests of what a session
launches, and on which buffers, without a device.

Every method of the real class runs (argument order and checks included); only the shared
library behind it is replaced.  Addresses come from one counter and are never reused, so an
argument of a logged call names its buffer for good; `live` holds the ranges not freed yet.
"""
import ctypes as C
import weakref

from karume_amd import _ffi
from karume_amd.runtime import GpuContext

_next_address = 1 << 20


class _Library:
    def __init__(self, gpu):
        self._gpu = gpu

    def __getattr__(self, name):
        if name not in _ffi.PROTOTYPES:
            raise AttributeError(name)
        special = getattr(self, "_" + name, None) if not name.startswith("_") else None
        gpu = self._gpu

        def call(*args):
            if special is not None:
                return special(*args)
            gpu.queue(name, args)
            return 0
        return call

    def _krm_buf_alloc(self, _handle, nbytes, out):
        global _next_address
        if sum(self._gpu.live.values()) + nbytes > self._gpu.memory:
            return -2
        out._obj.value = _next_address
        self._gpu.live[_next_address] = nbytes
        _next_address += (nbytes + 511) // 256 * 256
        return 0

    def _krm_last_error(self, _handle):
        return b"out of memory"

    def _krm_buf_free(self, _handle, address):
        del self._gpu.live[int(address)]
        return 0

    def _krm_attention_state_workspace(self, batch, heads, _kv_heads, _rows, depth, _window,
                                       max_past, _max_query, out):
        out._obj.value = batch * heads * (max_past // 64 + 1) * (depth + 2) * 4
        return 0

    def _krm_graph_begin(self, _handle):
        self._gpu.recording = []
        return 0

    def _krm_graph_end(self, _handle, out):
        self._gpu.graphs.append(self._gpu.recording)
        self._gpu.recording = None
        out._obj.value = len(self._gpu.graphs)
        return 0

    def _krm_graph_launch(self, _handle, graph):
        calls = self._gpu.graphs[graph.value - 1]
        assert calls is not None, "a destroyed graph was launched"
        self._gpu.log += calls
        return 0

    def _krm_graph_destroy(self, _handle, graph):
        self._gpu.graphs[graph.value - 1] = None
        return 0


class StandInGpu(GpuContext):
    def __init__(self):
        self._lib = _Library(self)
        self._handle = C.c_void_p(1)
        self.device = 0
        self._buffers = set()
        self.spare_holders = weakref.WeakSet()
        self.memory = 1 << 40
        self.live, self.graphs = {}, []
        self.log, self.recording = [], None

    def queue(self, name, args):
        (self.log if self.recording is None else self.recording).append((name, args[1:]))

    def clear(self):
        self.log = []

    def mentions(self, buffer):
        """Whether a logged call was given an address inside `buffer`."""
        inside = range(buffer.address, buffer.address + max(1, buffer.nbytes))
        return any(isinstance(a, int) and a in inside for _, args in self.log for a in args)

    def open_graphs(self):
        return sum(calls is not None for calls in self.graphs)
