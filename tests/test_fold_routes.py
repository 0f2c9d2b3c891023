"""Which plans are folded, and that the others are answered as well: COPY tensors sliced on a
part of their edges, or by two groups."""

import numpy as np
import pytest
from emulated import EmulatedAPI

from oracle import numpy_oracle
from tensororder_amd import _lib, fold, hip_api, network, plan_io, planners
from tensororder_amd.formula import parse_dimacs_text
from tensororder_amd.instances import random_3cnf
from tensororder_amd.network import BuiltTensor, TensorNetwork, VariableTensor
from tensororder_amd.plan import SlicedExecutionPlan
from tensororder_amd.tree import TreeContext


def _plan(n, seed):
    net = network.cnf_count(parse_dimacs_text(random_3cnf(n, int(1.9 * n), seed, True), "cachet"))
    return planners.best_plan(net, "factor", solver=None, seed=seed)


def _sliced_on(plan, groups):
    doc = plan_io.plan_to_dict(plan)
    doc["groups_to_slice"] = [sorted(int(e) for e in g) for g in groups]
    return doc


@pytest.mark.parametrize("seed", range(4))
@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_copies_sliced_on_a_part_of_their_edges(seed, et, tol):
    plan = _plan(12, seed)
    edge = plan.next_edge_to_slice
    whole = sorted(plan.network.find_equivalent_edges(edge))
    assert len(whole) > 1
    other = next(e for e in range(plan.network.num_edges()) if e not in whole and
                 len(plan.network.find_equivalent_edges(e)) > 1)
    cases = [[whole], [[edge]], [whole[:1], whole[1:]], [whole, [other]]]
    for groups in cases:
        doc = _sliced_on(plan, groups)
        want = numpy_oracle.contract_sliced(doc)
        api = EmulatedAPI(et)
        got = plan_io.plan_from_dict(doc)
        assert fold.has_copies(api._plan_inputs(got, None)[2]) == (groups == [whole])
        assert api.contract_sliced(got) == pytest.approx(want, rel=tol)


@pytest.mark.parametrize("et", [_lib.TO_F64, _lib.TO_F32S])
def test_groups_that_only_ones_hold(et):
    # two unweighted COPY tensors that share an edge, beside two that a weight is on: slicing the
    # first edge changes no value, but each slice counts
    net = TensorNetwork()
    ends = [net.add_node(VariableTensor(1, *w)) for w in ((1, 1), (1, 1), (0.3, 0.6), (1, 1))]
    net.connect(*ends[0][0], *ends[1][0])
    net.connect(*ends[2][0], *ends[3][0])
    ctx, tree = TreeContext(), None
    for end in ends:
        leaf = ctx.leaf(net, end[0][0])
        tree = leaf if tree is None else ctx.join(tree, leaf)
    plan = SlicedExecutionPlan(ctx.get_tree(tree), net)
    for groups, limit, want in (([], None, 1.8), ([{0}], None, 1.8), ([{0}], 1, 0.9), ([{1}], None, 1.8),
                                ([{1}], 1, 1.2), ([{0}, {1}], None, 1.8), ([{0}, {1}], 2, 0.9)):
        plan.groups_to_slice = groups
        exe = EmulatedAPI(et).prepare(plan, limit)
        got = exe.run()
        assert got.value == pytest.approx(want, rel=1e-6) and got.slices == exe.total == (limit or 2 ** len(groups))


def _star(n):
    """A plan of dense tensors and COPY tensors that opens 2 n variables before it sums any."""
    net, first, second = TensorNetwork(), [], []
    for _ in range(n):
        a, b, d = (net.add_node(BuiltTensor(np.ones((2, 2)))) for _ in range(3))
        c = net.add_node(VariableTensor(2, 1, 1))
        net.connect(*a[0], *c[0])
        net.connect(*c[1], *b[0])
        net.connect(*a[1], *d[0])
        net.connect(*d[1], *b[1])
        first += [a[0][0], c[0][0], d[0][0]]
        second.append(b[0][0])
    ctx, tree = TreeContext(), None
    for t in first + second:
        tree = ctx.leaf(net, t) if tree is None else ctx.join(tree, ctx.leaf(net, t))
    return SlicedExecutionPlan(ctx.get_tree(tree), net)


def _answer(call, plan):
    """What a call answers, with its kind of refusal in place of an answer."""
    try:
        return call(plan)
    except Exception as e:
        return type(e)


@pytest.mark.parametrize("n", [40, 600])
@pytest.mark.parametrize("et", [_lib.TO_F64, _lib.TO_F32S])
def test_far_too_large_plans_are_refused_alike(n, et, monkeypatch):
    # (a join over more variables than a float has exponents)
    plan, api = _star(n), EmulatedAPI(et)
    calls = [lambda p: api.contract_sliced(p), lambda p: api.contract_batch([p])]
    folded = [_answer(call, plan) for call in calls]
    monkeypatch.setattr(fold, "has_copies", lambda tables: False)
    assert folded == [_answer(call, plan) for call in calls] == [MemoryError] * 2


@pytest.mark.parametrize("esize", [8, 4])
def test_tensors_beyond_32_bit_offsets_run_edge_by_edge(esize):
    class Api:
        _esize, _regroup, _max_batch = esize, True, 64

        def _budget(self):
            return 1 << 50

    seen = set()
    for n in range(14, 21):
        _, tree, tables, _ = EmulatedAPI._plan_inputs(EmulatedAPI(heap_bytes=64), _star(n), None)
        folded = fold.analyse(tree, tables, esize, regroup=False)
        rank = max(t.rank for t in folded[0])
        folds = rank <= 32
        seen.add(rank)
        assert hip_api.HipAPI.choose_folded_batch(Api(), folded, tree, tables, 1) == folds
        assert (fold.analyse_batch([(tree, tables)], esize, regroup=False) is not None) == folds
        if folds:  # every record of the plan holds its offsets
            nodes = folded[0]
            for t in nodes:
                t.ptr = t.bstride = 0
            for t in nodes:
                if not t.is_leaf and t.geom["var"]["kind"] == "fold":
                    scratch = {"partial": (0, 0)}
                    for record in fold.join_records(t, nodes, 1, esize, False, 0, scratch, lambda n: 0, (0, 0)):
                        assert bytes(record[4])
    assert 32 in seen and max(seen) > 32


def test_exponents_of_programs_fit(monkeypatch):
    # a program's records hold 32-bit exponents, to which a node adds less than 2^11
    assert fold.EXPONENT_NODES * 2 ** 11 <= 2 ** 31
    plan = _plan(12, 0)
    want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
    for et, folds in ((_lib.TO_F64, True), (_lib.TO_F32S, False)):
        api = EmulatedAPI(et)
        _, tree, tables, _ = api._plan_inputs(plan, None)
        nodes = fold.analyse(tree, tables, api._esize)[0]
        for most, fits in ((len(nodes), True), (len(nodes) - 1, folds)):
            monkeypatch.setattr(fold, "EXPONENT_NODES", most)
            assert (fold.analyse_batch([(tree, tables)], api._esize) is not None) == fits
            exe = api.prepare(plan)
            assert (exe.prog.host_accum is not None) == fits  # (the walk's sums stay on the device)
            assert exe.run().value == pytest.approx(want, rel=1e-6)
