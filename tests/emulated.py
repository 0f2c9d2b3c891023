"""The executor's host code over the emulator: a ``HipAPI`` whose device memory is the emulated
heap and whose launches run in numpy, so that routes, runs and executables' lives can be tested
without a GPU.  Launches run as they are queued; ``synchronize`` and ``finish`` only count."""

import contextlib
import ctypes
import math
import types

import emulator
import numpy as np
from test_fold import FoldEmulator, _spread

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
    """... with the bookkeeping launches that open a run of the edge walk, sums that also go to
    host memory, and results of more than two operands scaled by their own largest entry."""

    def _tree_task(self, d, op, chunk, batch, data, recs, pending):
        if not self.scaled or int(op[0]) >> 16 & 3 < 2:
            return super()._tree_task(d, op, chunk, batch, data, recs, pending)
        head = int(op[0])
        lo, lk, nloop = head & 15, head >> 4 & 15, head >> 8 & 15
        prod, e = 1.0, 0
        for j in range((head >> 16 & 3) + 1):
            bits = op[64 + 16 * j:80 + 16 * j]
            k = (_spread(bits, lo, lk)[:, None] + _spread(bits, 6, nloop)[None, :]).ravel()
            idx = _spread(bits, 0, lo)[:, None] + k[None, :]
            addr, slot = int(op[1 + 2 * j]) | int(op[2 + 2 * j]) << 32, int(op[16 + j])
            if head >> (20 + j) & 1:
                prod = prod * data[addr + idx].astype(np.float64)
                e += recs[slot][0]
            else:
                src = self.heap.view(addr + batch * int(op[11 + j]) * 4, np.float32, int(idx.max()) + 1)
                prod = prod * src[idx].astype(np.float64)
                e += self.get_rec(d.recs, slot + (batch if head >> (25 + j) & 1 else 0))[0]
        total = prod.sum(axis=1)
        x = math.frexp(np.abs(total).max())[1]
        v = np.ldexp(total, -x).astype(np.float32)
        o, addr, slot = _spread(op[32:48], 0, lo), int(op[9]) | int(op[10]) << 32, int(op[20])
        self.operands = getattr(self, "operands", set()) | {(head >> 16 & 3) + 1}

        def write():
            m = np.abs(v).max()
            if head >> 24 & 1:
                data[addr + o] = v
                recs[slot][:] = [e + x, float(m)]
            else:
                self.heap.view(addr + batch * int(op[15]) * 4, np.float32, int(o.max()) + 1)[o] = v
                self.set_rec(d.recs, slot + (batch if head >> 29 & 1 else 0), exp=e + x, maxbits=int(m.view(np.uint32)))
        pending.append(write)

    def op_4(self, L):
        if not L.variant & _lib.TO_FINISH_NORM:
            return super().op_4(L)
        assert self.scaled
        for i in range(L.count):
            d = self.heap.read_struct(_lib.JoinDesc, L.descs + i * ctypes.sizeof(_lib.JoinDesc))
            assert d.partial in self.gemm_partials and d.fx == d.fy == 0
            P = self.heap.view(d.partial, np.float64, d.nbatch * d.nsplit).reshape(-1, d.nsplit)
            for b, total in enumerate(P.sum(axis=1)):
                m, x = math.frexp(total)
                e = x + sum(exp + emulator._scale_exp(top) for exp, top in
                            (self.get_rec(d.xs, b * d.xsb), self.get_rec(d.ys, b * d.ysb)))
                self.heap.view(d.c + 4 * b * d.cb, np.float32, 1)[0] = m
                self.set_rec(d.cs, b, exp=e, maxbits=int(np.float32(abs(m)).view(np.uint32)))

    def op_6(self, L):
        if L.variant == 0:
            return emulator.Emulator.op_6(self, L)
        device = _lib.Launch.from_buffer_copy(bytes(L))
        device.iaux1 = 0
        sums = self.heap.read_struct(_lib.Accum, L.aux2).pad  # written so far
        super().op_6(device)
        acc = self.heap.read_struct(_lib.Accum, L.aux2)
        acc.pad = sums + bool(L.iaux1)
        self.heap.view(L.aux2, "u1", ctypes.sizeof(acc))[:] = list(bytes(acc))
        if L.iaux1:
            ctypes.memmove(L.iaux1, bytes(acc), ctypes.sizeof(acc))

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
        self._lib = types.SimpleNamespace(to_wait=lambda *a: _lib.TO_OK, 
                                          to_wall_clock_khz=lambda khz: setattr(khz._obj, "value", 1) or _lib.TO_OK)
        self.budget, self.waits, self.fail_at = 1 << 40, 0, None

    def _alloc(self, nbytes):
        return _Device(self.heap.alloc(max(1, int(nbytes))))

    def _alloc_host(self, nbytes):
        return _Host(nbytes)

    def prepare_batch(self, plans):
        self._alloc_host = self._alloc  # (a batch reads its accumulators as tensors)
        try:
            return super().prepare_batch(plans)
        finally:
            del self._alloc_host

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
