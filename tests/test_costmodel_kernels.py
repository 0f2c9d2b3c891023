"""The plan-cost model's kernels at the edges of their row tiles, and with buffers that are not
16-byte aligned, against the float64 oracle."""

import ctypes

import numpy as np
import pytest

from oracle import mlp_oracle
from tensororder_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 127, 129, 513, 2050])
@pytest.mark.parametrize("shift", [0, 1])
def test_rows_and_alignment(n, shift):
    import torch

    print("case mlp rows", n, "shift", shift, flush=True)
    lib = _lib.load()
    rng = np.random.default_rng(n)
    p = (rng.standard_normal(_lib.MLP_NPARAMS) * 0.3).astype(np.float32)
    x = rng.standard_normal((n, 16)).astype(np.float32)
    t = rng.standard_normal((n, 2)).astype(np.float32)

    def dev(a):  # a device copy, its first entry `shift` floats after an aligned address
        buf = torch.full((a.size + shift,), float("nan"), dtype=torch.float32, device="cuda")
        buf[shift:] = torch.from_numpy(np.ascontiguousarray(a, np.float32).ravel()).cuda()
        return buf

    def ptr(buf):
        return ctypes.c_void_p(buf.data_ptr() + 4 * shift)

    nan = np.full
    P, X, T = dev(p), dev(x), dev(t)
    H1, H2, DH1, DH2 = (dev(nan((n, 64), np.nan)) for _ in range(4))
    Y, DY = dev(nan((n, 2), np.nan)), dev(nan((n, 2), np.nan))
    G, L = dev(nan(_lib.MLP_NPARAMS, np.nan)), dev(nan(1, np.nan))
    torch.cuda.synchronize()
    _lib.check(lib.to_mlp_forward(ptr(P), ptr(X), n, ptr(H1), ptr(H2), ptr(Y), None), "to_mlp_forward")
    _lib.check(lib.to_mlp_backward(ptr(P), ptr(X), ptr(H1), ptr(H2), ptr(Y), ptr(T), n, ptr(DY), ptr(DH2), ptr(DH1),
                                   ptr(G), ptr(L), None), "to_mlp_backward")
    torch.cuda.synchronize()
    _, _, want = mlp_oracle.forward(p.astype(np.float64), x)
    loss, grad = mlp_oracle.loss_and_grad(p.astype(np.float64), x, t)
    # sums of at most 64 float terms of order 1 per layer, the row sums in double
    np.testing.assert_allclose(Y[shift:].cpu().numpy().reshape(n, 2), want, rtol=1e-4, atol=1e-5)
    assert float(L[shift]) == pytest.approx(loss, rel=1e-5)
    scale = np.abs(grad).max()
    np.testing.assert_allclose(G[shift:].cpu().numpy(), grad, rtol=1e-3, atol=1e-5 * scale)
    # both in one call: the same numbers
    G1, L1 = dev(nan(_lib.MLP_NPARAMS, np.nan)), dev(nan(1, np.nan))
    outs = [dev(nan((n, w), np.nan)) for w in (64, 64, 2, 2, 64, 64)]
    torch.cuda.synchronize()
    _lib.check(lib.to_mlp_gradient(ptr(P), ptr(X), ptr(T), n, *map(ptr, outs), ptr(G1), ptr(L1), None), "to_mlp_gradient")
    torch.cuda.synchronize()
    for got, ref in zip(outs + [G1, L1], (H1, H2, Y, DY, DH2, DH1, G, L)):
        np.testing.assert_allclose(got[shift:].cpu().numpy(), ref[shift:].cpu().numpy(), rtol=1e-5,
                                   atol=1e-6 * float(ref[shift:].abs().max()))


def test_training_rows_are_there_when_they_are_read():
    # the rows of a batch are gathered where the kernels that read them run, not on the caller's
    # stream, which may be busy
    import torch

    from tensororder_amd import costmodel
    from tensororder_amd.hip_api import HipAPI

    rng = np.random.default_rng(1)
    x = rng.standard_normal((600, 16))
    y = np.stack([x[:, 0] + x[:, 1], x[:, 2]], axis=1)
    got = []
    for busy in (False, True):
        model = costmodel.CostModel(HipAPI(), seed=5)
        print("case training, caller's stream busy:", busy, flush=True)
        a = torch.rand((4096, 4096), device="cuda")
        pending = []
        select = torch.Tensor.index_select

        def after_work(t, *args):  # a product before every gather, on the stream it runs on
            if busy:
                with torch.cuda.stream(torch.cuda.default_stream()):
                    pending.append(a @ a)
            return select(t, *args)

        torch.Tensor.index_select = after_work
        try:
            got.append(model.fit(x, y, epochs=3, batch=128))
        finally:
            torch.Tensor.index_select = select
        torch.cuda.synchronize()
    assert got[0] == got[1]


def test_rows_beyond_one_launch():
    # 2^27 rows and some: more threads, at 32 a row, than a launch counts
    import torch

    n = (1 << 27) + 11
    free, _ = torch.cuda.mem_get_info()
    if free < 600 * n + (8 << 30):
        pytest.skip("needs %d GB of device memory" % (600 * n >> 30))
    print("case mlp rows", n, flush=True)
    lib = _lib.load()
    rng = np.random.default_rng(0)
    p = (rng.standard_normal(_lib.MLP_NPARAMS) * 0.3).astype(np.float32)
    few = 64
    x = rng.standard_normal((few, 16)).astype(np.float32)
    P, X = torch.from_numpy(p).cuda(), torch.zeros((n, 16), dtype=torch.float32, device="cuda")
    at = [0, (1 << 26) - few // 2, n - few]  # across the ends of the launches
    for r in at:
        X[r:r + few] = torch.from_numpy(x).cuda()
    H1, H2 = (torch.empty((n, 64), dtype=torch.float32, device="cuda") for _ in range(2))
    Y = torch.full((n, 2), float("nan"), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    _lib.check(lib.to_mlp_forward(*(ctypes.c_void_p(t.data_ptr()) for t in (P, X)), n,
                                  *(ctypes.c_void_p(t.data_ptr()) for t in (H1, H2, Y)), None), "to_mlp_forward")
    torch.cuda.synchronize()
    _, _, want = mlp_oracle.forward(p.astype(np.float64), x)
    for r in at:
        np.testing.assert_allclose(Y[r:r + few].cpu().numpy(), want, rtol=1e-4, atol=1e-5)
    assert not bool(torch.isnan(Y).any())
    del X, H1, H2, Y
    torch.cuda.empty_cache()
