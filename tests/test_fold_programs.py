"""How the programs of a plan are cut: to what LDS holds, with work that grows with the plan, and
to the same count wherever the cuts lie."""

import numpy as np
import pytest
import test_fold
from emulated import EmulatedAPI

from oracle import numpy_oracle
from tensororder_amd import _lib, fold, network, plan_io, planners, schedule
from tensororder_amd.formula import parse_dimacs_text
from tensororder_amd.network import BuiltTensor, TensorNetwork, VariableTensor
from tensororder_amd.tree import TreeContext


def grid_plan(width, length):
    """The line plan of a vertex cover of a width x length grid."""
    def v(i, j):
        return i * width + j + 1

    clauses = [(v(i, j), v(i, j + 1)) for i in range(length) for j in range(width - 1)]
    clauses += [(v(i, j), v(i + 1, j)) for i in range(length - 1) for j in range(width)]
    text = "p cnf %d %d\n" % (width * length, len(clauses)) + "".join("%d %d 0\n" % c for c in clauses)
    return planners.best_plan(network.cnf_count(parse_dimacs_text(text, "cachet")), "line", solver=None, seed=0)


def chain(n):
    """(tree, tables) of a product of n 2 x 2 matrices, COPY tensors between them."""
    net, order, last = TensorNetwork(), [], None
    for i in range(n):
        ends = net.add_node(BuiltTensor(np.ones((2,) * (1 if i in (0, n - 1) else 2))))
        if last is not None:
            tie = net.add_node(VariableTensor(2, 1, 1))
            net.connect(*last, *tie[0])
            net.connect(*tie[1], *ends[0])
            order.append(tie[0][0])
        order.append(ends[0][0])
        last = ends[-1]
    ctx, tree, tables = TreeContext(), None, {}
    for t in order:
        rank = net[t].rank
        tables[t] = schedule.LeafTable(np.eye(2).reshape(1, -1) if rank == 2 else np.ones((1, 2)), [], rank,
                                       copy=(1, 1, True) if isinstance(net[t], VariableTensor) else None)
        tree = ctx.leaf(net, t) if tree is None else ctx.join(tree, ctx.leaf(net, t))
    return ctx.get_tree(tree), tables


def checked_programs(nodes, W, esize, lds=None):
    """The programs of a plan, and how many joins were looked at to find them."""
    seen = []
    inner = fold._program

    def counted(*args):
        p = inner(*args)
        seen.append(len(p.members))
        return p

    fold._program = counted
    try:
        programs = fold.tree_programs(nodes, W, esize, esize == 4, lds)
    finally:
        fold._program = inner
    members = [i for p in programs for i in p.members]
    assert len(members) == len(set(members))
    assert all(p.lds <= (lds or fold.TREE_LDS) for p in programs)
    return programs, sum(seen)


@pytest.mark.parametrize("esize", [8, 4])
@pytest.mark.parametrize("name", ["grid", "chain"])
def test_long_plans_are_cut_with_little_work(name, esize):
    if name == "grid":
        tree, tables = test_fold.plan_inputs(grid_plan(8, 120))[1:3]
    else:
        tree, tables = chain(40000 if esize == 4 else 8000)
    nodes, _ = fold.analyse(tree, tables, esize)
    fold.choose_all(nodes, 1, esize)
    programs, seen = checked_programs(nodes, 1, esize)
    joins = sum(not n.is_leaf for n in nodes)
    assert joins > 2500 and seen < 16 * joins
    if name == "chain" and esize == 4:
        assert 2 < len(programs) < 10  # (the records of a program's tensors fill LDS)
    # next to all joins are in programs: what does not fit one goes on in another
    assert sum(len(p.members) for p in programs) > 0.99 * joins
    assert len(fold.phase_groups(nodes, False, "level", programs)) < 8


@pytest.mark.parametrize("lds", [64, 256, 1024, 8192])
@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_counts_wherever_programs_are_cut(lds, et, tol, monkeypatch):
    monkeypatch.setattr(fold, "TREE_LDS", lds)
    monkeypatch.setattr(fold, "TREE_LONG", 8)
    for kind, n, slices in (("vc", 30, 1), ("cnf", 20, 2)):
        plan = test_fold._formula_plan(kind, n, 3, slices)
        want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
        got, prog, _ = test_fold.emulate(plan, et, 1 << slices)
        assert got == pytest.approx(want, rel=tol, abs=0)
        assert len(prog.programs) > 2
        checked_programs(prog.nodes, 1 << slices, 8 if et == _lib.TO_F64 else 4)


@pytest.mark.parametrize("most", [1, 3, 40])
@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_programs_hold_no_more_products_than_a_task_names(most, et, tol, monkeypatch):
    assert fold.TREE_PRODUCTS == 0xffff + 1  # bits 0-15 of a task
    monkeypatch.setattr(fold, "TREE_PRODUCTS", most)
    plan = test_fold._formula_plan("vc", 40, 1, 0)
    want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
    got, prog, _ = test_fold.emulate(plan, et, 1)
    assert got == pytest.approx(want, rel=tol, abs=0)
    sizes = [sum(map(len, p.levels)) for p in prog.programs]
    assert max(sizes) <= most and len(sizes) > 1
    tree, tables = chain(500)
    nodes, _ = fold.analyse(tree, tables, 8)
    fold.choose_all(nodes, 1, 8)
    programs, _ = checked_programs(nodes, 1, 8)
    assert max(sum(map(len, p.levels)) for p in programs) <= most
    monkeypatch.setattr(fold, "TREE_PRODUCTS", 0)
    with pytest.raises(ValueError):
        fold.tree_words(programs[0], nodes, 16, lambda n: 0, (0, 0))


@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_the_layout_of_the_accepted_batch_is_compiled(et, tol, monkeypatch):
    # forms and programs are made once for each batch size tried, and are those of the last
    plan = test_fold._formula_plan("cnf", 16, 1, 6)
    want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
    made, seen = [], set()
    inner = fold.choose_all
    monkeypatch.setattr(fold, "choose_all", lambda nodes, W, *a: made.append(W) or inner(nodes, W, *a))
    for share in (1.0, 0.6, 0.3):
        api = EmulatedAPI(et)
        total, tree, tables, groups = api._plan_inputs(plan, None)
        esize = api._esize
        nodes = fold.analyse(tree, tables, esize)[0]
        fixed = sum(t.size for t in tables.values()) * esize
        one = schedule.peak_bytes(schedule.analyse(tree, tables), tables, 1, et)  # (below, it is refused)
        api.budget = fixed + max(int(share * fold.peak_bytes(nodes, 64, esize)), one)
        made.clear()
        exe = api.prepare(plan)
        assert made == sorted(made, reverse=True) and len(set(made)) == len(made)
        assert made[0] == 64 and exe.prog.nbatch == made[-1]
        seen.add(made[-1])
        assert exe.run().value == pytest.approx(want, rel=tol, abs=0)
    assert len(seen) > 1
    # a shape tuned in between is a new layout
    api = EmulatedAPI(et)
    api._tune = lambda nodes, W: 1
    made.clear()
    assert api.contract_sliced(plan) == pytest.approx(want, rel=tol, abs=0)
    assert made == [64, 64]


def test_analysis_of_many_weights_is_linear(monkeypatch):
    # weights of variables that no clause holds are scalars, and multiply one leaf: which one is
    # looked for once, not among all leaves for each
    n = 1200
    lines = ["p cnf %d %d" % (2 * n, n - 1)] + ["%d %d 0" % (i, i + 1) for i in range(1, n)]
    lines += ["w %d 0.25" % i for i in range(1, 2 * n + 1)]
    net = network.cnf_count(parse_dimacs_text("\n".join(lines) + "\n", "cachet"))
    tree, tables = test_fold.plan_inputs(planners.best_plan(net, "line", solver=None, seed=0))[1:3]
    compared = [0]

    def counted(values, *args, **kw):
        values = list(values)
        compared[0] += len(values)
        return min(values, *args, **kw)

    monkeypatch.setattr(fold, "min", counted, raising=False)
    nodes, _ = fold.analyse(tree, tables, 8)
    assert len(nodes) > 2 * n and compared[0] < 40 * len(nodes)


@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_weights_reach_a_wide_clause_together(et, tol):
    # two clauses of 14 literals over 24 variables, and variables that none holds: a leaf takes the
    # weights of all its variables in few joins, no more than the walk takes
    first, second = range(1, 15), range(11, 25)
    lines = ["p cnf 30 2"] + [" ".join(str(v * (-1) ** (v % 3)) for v in c) + " 0" for c in (first, second)]
    lines += ["w %d %r" % (v, 0.2 + v / 60) for v in range(1, 31)]
    net = network.cnf_count(parse_dimacs_text("\n".join(lines) + "\n", "cachet"))
    for planner in ("line", "factor"):
        plan = planners.best_plan(net, planner, solver=None, seed=0)
        tree, tables = test_fold.plan_inputs(plan)[1:3]

        def large(nodes):
            return sum(max(nodes[n.left].rank, nodes[n.right].rank) >= fold.BIG_RANK for n in nodes if not n.is_leaf)

        esize = 8 if et == _lib.TO_F64 else 4
        assert large(fold.analyse(tree, tables, esize)[0]) <= max(6, large(schedule.analyse(tree, tables)))
        want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
        assert EmulatedAPI(et).contract_sliced(plan) == pytest.approx(want, rel=tol)
