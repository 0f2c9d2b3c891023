"""The executor's host code over the emulator: a ``HipAPI`` whose device memory is the emulated
heap and whose launches run in numpy, so that routes, runs and executables' lives can be tested
without a GPU.  Launches run as they are queued; ``synchronize`` and ``finish`` only count."""

import contextlib
import ctypes
import types

import emulator
from test_fold import FoldEmulator

from tensororder_amd import _lib, hip_api


class _Host:
    """Host memory that the device writes."""

    def __init__(self, nbytes):
        self.mem = (ctypes.c_char * max(1, int(nbytes)))()

    def data_ptr(self):
        return ctypes.addressof(self.mem)


class _Copied:
    def __init__(self, array):
        self.array = array

    def cpu(self):
        return self

    def numpy(self):
        return self.array


class _Device:
    def __init__(self, buf):
        self.buf = buf

    def data_ptr(self):
        return self.buf.data_ptr()

    def __getitem__(self, sl):
        return _Copied(self.buf[sl])


class RunEmulator(FoldEmulator):
    """... with the bookkeeping launches that open a run of the edge walk, and sums that also go
    to host memory."""

    def op_6(self, L):
        if L.variant == 0:
            return emulator.Emulator.op_6(self, L)
        device = _lib.Launch.from_buffer_copy(bytes(L))
        device.iaux1 = 0
        super().op_6(device)
        acc = self.heap.read_struct(_lib.Accum, L.aux2)
        acc.pad += 1
        raw = bytes(acc)
        self.heap.view(L.aux2, "u1", len(raw))[:] = list(raw)
        if L.iaux1:
            ctypes.memmove(L.iaux1, raw, len(raw))
            if L.variant == 1 and acc.pad:
                self.sums = getattr(self, "sums", 0) + 1

    def op_8(self, L):
        self.heap.view(L.aux2, "u1", ctypes.sizeof(_lib.Accum))[:] = 0
        self.heap.view(L.aux3, "i8", 1)[0] = 0


class EmulatedAPI(hip_api.HipAPI):
    def __init__(self, entry_type=_lib.TO_F64, max_batch=1 << 16, heap_bytes=1 << 28, emulate=RunEmulator):
        self.heap = emulator.Heap(heap_bytes)
        self.emulator = emulate(self.heap, entry_type)
        self._entry_type, self._max_batch = entry_type, max_batch
        self._use_graph, self._regroup, self._autotune, self._device_leaves = False, True, False, True
        self._stream = types.SimpleNamespace(cuda_stream=0)
        self._torch = types.SimpleNamespace(cuda=types.SimpleNamespace(stream=lambda s: contextlib.nullcontext()))
        self._lib = types.SimpleNamespace(to_wait=lambda *a: _lib.TO_OK)
        self.budget, self.waits, self.fail_at = 1 << 40, 0, None

    def _alloc(self, nbytes):
        return _Device(self.heap.alloc(max(1, int(nbytes))))

    def _alloc_host(self, nbytes):
        return _Host(nbytes)

    def _upload(self, dst, host_bytes):
        self.heap.write(dst, host_bytes)

    def _run(self, launches):
        for L in launches:
            if self.fail_at is not None:
                if self.fail_at == 0:
                    self.fail_at = None
                    raise KeyboardInterrupt
                self.fail_at -= 1
            self.emulator.run([L])

    def _budget(self):
        return self.budget

    def synchronize(self):
        self.waits += 1

    finish = synchronize
