"""to_tensordot's 16-byte streamed form at the edges of its rule (every y chunk, shared axes
next to the lowest bits, the smallest sizes it takes and those just below, tensors that are not
16-byte aligned) against numpy, and to_upload's sizes."""

import ctypes

import numpy as np
import pytest

from tensororder_amd import _lib

pytestmark = pytest.mark.gpu

# (rank a, rank b, a's shared axes counted from the last, shift of a and c in entries)
CASES = [(20, 0, [], 0), (19, 1, [], 0), (20, 3, [3], 0), (19, 4, [3, 18], 0), (18, 6, [2, 5, 9], 0), (18, 8, [4, 3, 17, 10], 0),
         (17, 7, [2, 3, 4], 0), (20, 3, [0], 0), (20, 3, [1], 0), (18, 3, [2], 0), (20, 5, [3, 7], 1), (20, 5, [3, 7], 2)]


@pytest.mark.parametrize("et", ["f64", "f32s"])
@pytest.mark.parametrize("ra,rb,low,shift", CASES)
def test_streamed_forms(et, ra, rb, low, shift):
    import torch

    print("case tensordot form", et, ra, rb, low, shift, flush=True)
    lib = _lib.load()
    dt = np.float64 if et == "f64" else np.float32
    rng = np.random.default_rng(ra * 100 + rb)
    s = len(low)
    la = [ra - 1 - p for p in low]
    lb = [int(x) for x in rng.permutation(rb)[:s]]
    a, b = rng.uniform(0.25, 1.0, (2,) * ra).astype(dt), rng.uniform(0.25, 1.0, (2,) * rb).astype(dt)
    want = np.tensordot(a.astype(np.float64), b.astype(np.float64), (la, lb)).ravel()

    def dev(x):
        t = torch.full((x.size + shift,), float("nan"), dtype=torch.float64 if et == "f64" else torch.float32, device="cuda")
        t[shift:] = torch.from_numpy(np.ascontiguousarray(x).ravel()).cuda()
        return t

    ta, tb, tc = dev(a), dev(b), dev(np.full(want.size, np.nan))
    recs = torch.tensor([[0, int(np.float32(1.0).view(np.uint32))]] * 3, dtype=torch.int64, device="cuda")
    ax = [(ctypes.c_int32 * max(1, s))(*v) for v in (la, lb)]
    p, off = ctypes.c_void_p, shift * a.itemsize
    torch.cuda.synchronize()
    _lib.check(lib.to_tensordot(p(ta.data_ptr() + off), p(tb.data_ptr() + off), p(tc.data_ptr() + off), ra, rb,
                                ctypes.addressof(ax[0]), ctypes.addressof(ax[1]), s,
                                _lib.TO_F64 if et == "f64" else _lib.TO_F32S, p(recs[0].data_ptr()), p(recs[1].data_ptr()),
                                p(recs[2].data_ptr()), None, 0, None), "to_tensordot")
    torch.cuda.synchronize()
    got = tc[shift:].cpu().numpy().astype(np.float64)
    if et == "f64":
        np.testing.assert_allclose(got, want, rtol=1e-14)
    else:  # double sums of exact products, one rounding at the store
        np.testing.assert_allclose(got * 2.0 ** int(recs[2, 0]), want, rtol=1.2e-7)
        assert int(recs[2, 1]) & 0xffffffff == int(np.float32(got.max()).view(np.uint32))


# float joins with shared ranges so long that the general form's slab of double y entries holds
# only a part of the 2^fy of them (2^10 by 8, 2^11 by 4, 2^12 by 2), and the next shorter ones,
# where it holds all
LONG = [(24, 13, 10), (25, 13, 11), (26, 13, 12), (24, 12, 9), (25, 12, 10), (26, 12, 11)]


@pytest.mark.parametrize("ra,rb,s", LONG)
def test_long_shared_ranges(ra, rb, s):
    test_streamed_forms("f32s", ra, rb, list(range(2, 2 + s)), 0)


@pytest.mark.parametrize("words", [0, 1, 767, 768, 769, 5000])
def test_upload(words):
    import torch

    lib = _lib.load()
    src = np.arange(words, dtype=np.uint32) * 2654435761
    dst = torch.zeros(words + 1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    assert lib.to_upload(ctypes.c_void_p(dst.data_ptr()), src.ctypes.data, 4 * words, None) == _lib.TO_OK
    src[:] = 0  # the host memory may be reused at once
    torch.cuda.synchronize()
    got = dst.cpu().numpy().view(np.uint32)
    np.testing.assert_array_equal(got[:words], np.arange(words, dtype=np.uint32) * 2654435761)
    assert got[words] == 0
    assert lib.to_upload(ctypes.c_void_p(dst.data_ptr()), src.ctypes.data, 3, None) == _lib.TO_ERR_INVALID
