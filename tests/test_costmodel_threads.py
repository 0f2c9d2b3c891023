"""Gradients of one plan-cost model taken by several threads at once: each gets its own loss."""

import ctypes
import threading
import types

import torch

from tensororder_amd import _lib, costmodel


def test_each_thread_reads_its_own_loss():
    both = threading.Barrier(2)
    model = object.__new__(costmodel.CostModel)
    model.losses = threading.local()
    model.params = model.grad = torch.zeros(1)
    model.torch = types.SimpleNamespace(float32=torch.float32, zeros=lambda n, dtype, pin_memory: torch.zeros(n, dtype=dtype))
    model._buffers = lambda n: [torch.zeros(1)] * 3
    # the device has written both losses before either thread reads
    model.api = types.SimpleNamespace(_stream=types.SimpleNamespace(cuda_stream=0), finish=lambda: both.wait(30))

    def gradient(params, x, target, n, *rest):
        loss = ctypes.cast(rest[-2], ctypes.POINTER(ctypes.c_float))
        loss[0] = float(n)
        return _lib.TO_OK

    model.lib = types.SimpleNamespace(to_mlp_gradient=gradient)
    got = {}

    def work(n):
        for _ in range(3):
            got.setdefault(n, []).append(model.gradient(torch.zeros(n, 16), torch.zeros(n, 2))[0])

    threads = [threading.Thread(target=work, args=(n,)) for n in (3, 5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got == {3: [3.0] * 3, 5: [5.0] * 3}
