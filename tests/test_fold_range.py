"""FP32-scaled folded plans whose numbers lie far apart: a product of several tensors, and a dot
product of two joins that are not stored, keep their bits where they are far below the product
of their operands' maxima."""

import ctypes

import numpy as np
import pytest
import test_fold
from emulated import EmulatedAPI

from oracle import numpy_oracle
from tensororder_amd import _lib, hip_api, network, plan_io, planners
from tensororder_amd.formula import parse_dimacs_text

# unit clauses against wide ones: the count is w^4, each tensor of the plan spans 1 to w
CLAUSES = ["1", "2", "3", "4", "1 2 3", "2 3 4"]
WEIGHTS = [1e-18, 1e-20, 1e-22, 1e-25]


def _plan(w, planner, n=4):
    """n variables in a row, forced true one by one and by threes: the count is w^n."""
    clauses = ["%d" % (i + 1) for i in range(n)] + ["%d %d %d" % (i + 1, i + 2, i + 3) for i in range(n - 2)]
    assert n != 4 or clauses == CLAUSES
    lines = ["p cnf %d %d" % (n, len(clauses))] + [c + " 0" for c in clauses]
    lines += ["w %d %r" % (i + 1, w) for i in range(n)]
    net = network.cnf_count(parse_dimacs_text("\n".join(lines) + "\n", "cachet"))
    return planners.best_plan(net, planner, solver=None, seed=0)


@pytest.mark.parametrize("w", WEIGHTS)
@pytest.mark.parametrize("planner", ["line", "factor"])
def test_small_weights_emulated(w, planner):
    for n in (4, 9):
        plan = _plan(w, planner, n)
        want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
        assert want == pytest.approx(w ** n, rel=1e-9, abs=0)
        api = EmulatedAPI(_lib.TO_F32S)
        exe = api.prepare(plan)
        got = exe.run()
        assert api.emulator.operands & {3, 4}  # products of several tensors are among them
        assert got.mant * 2.0 ** got.exp == pytest.approx(want, rel=1e-6, abs=0)


@pytest.mark.gpu
@pytest.mark.parametrize("w", WEIGHTS)
def test_small_weights_on_the_device(w):
    api = hip_api.HipF32API()
    plans = [_plan(w, planner, n) for planner in ("line", "factor") for n in (4, 9)]
    print("case small weights", w, flush=True)
    wants = [numpy_oracle.contract_sliced(plan_io.plan_to_dict(p)) for p in plans]
    got = []
    for p in plans:
        exe = api.prepare(p)
        got.append(exe.run().value)
        exe.close()
    np.testing.assert_allclose(got, wants, rtol=1e-6)
    np.testing.assert_allclose(api.contract_batch(plans), wants, rtol=1e-6)


class _Apart:
    """Random numbers of ``_pair``'s tensors, in the order it asks for them (large, small, large,
    small): the large ones hold numbers near 1 at entries where the other holds 0, and numbers
    near 1e-23 at those (by the two lowest variables) that meet."""

    def __init__(self, seed):
        self.rng, self.calls = np.random.default_rng(seed), 0

    def __getattr__(self, name):
        return getattr(self.rng, name)

    def uniform(self, lo, hi, shape):
        out = self.rng.uniform(lo, hi, shape)
        if self.calls % 2 == 0:
            low = np.arange(shape[1]) & 3
            out[:, low == (1 if self.calls else 0)] = 0.0
            out[:, low > 1] *= 1e-23
        self.calls += 1
        return out


# cases of every number of summed variables, with and without blocks sharing a sum
APART = [test_fold.PAIRS[i] for i in (0, 1, 3, 4, 5, 7, 8)]


@pytest.mark.parametrize("case", APART)
def test_dot_products_of_small_numbers_emulated(case):
    ptr = {}
    api = EmulatedAPI(_lib.TO_F32S)

    def alloc(n):
        b = api.heap.alloc(n)
        ptr[b.data_ptr()] = b
        return b.data_ptr()

    records, nodes, recs, want = test_fold._pair(case, _lib.TO_F32S, alloc, lambda at, data: api.heap.write(ptr[at], data),
                                                 _Apart(case[0]))
    assert abs(want).max() < 1e-36  # (most of it the exponents of 3 a tensor)
    api.emulator.run(test_fold._launches(records, alloc, lambda at, data: api.heap.write(ptr[at], data)))
    got = api.heap.view(nodes[-1].ptr, np.float32, case[5]).reshape(-1, 1)[:len(want)]
    rec = [api.heap.read_struct(_lib.ScaleRec, recs[nodes[-1].idx] + 16 * b) for b in range(len(want))]
    test_fold._check(case, _lib.TO_F32S, got, rec, want)


# (the last: whole blocks of slices, a sum in one block)
@pytest.mark.gpu
@pytest.mark.parametrize("case", APART + [test_fold.PAIRS[6]])
def test_dot_products_of_small_numbers_on_the_device(case):
    import torch

    print("case small dot", case, flush=True)
    api, ptr = hip_api.HipF32API(), {}

    def alloc(n):
        t = torch.full((n,), 255, dtype=torch.uint8, device="cuda")
        ptr[t.data_ptr()] = t
        return t.data_ptr()

    def write(at, data):
        ptr[at][:len(data)] = torch.frombuffer(bytearray(data), dtype=torch.uint8).cuda()

    records, nodes, recs, want = test_fold._pair(case, _lib.TO_F32S, alloc, write, _Apart(case[0]))
    launches = test_fold._launches(records, alloc, write)
    torch.cuda.synchronize()
    api._run(launches)
    api.synchronize()
    got = ptr[nodes[-1].ptr].cpu().numpy().view(np.float32).reshape(-1, 1)[:len(want)]
    raw = ptr[recs[nodes[-1].idx]].cpu().numpy().tobytes()
    size = ctypes.sizeof(_lib.ScaleRec)
    rec = [_lib.ScaleRec.from_buffer_copy(raw[size * b:size * b + size]) for b in range(len(want))]
    test_fold._check(case, _lib.TO_F32S, got, rec, want)
