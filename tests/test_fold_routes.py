"""Which plans are folded, and that the others are answered as well: COPY tensors sliced on a
part of their edges, or by two groups."""

import pytest
from emulated import EmulatedAPI

from oracle import numpy_oracle
from tensororder_amd import _lib, fold, network, plan_io, planners
from tensororder_amd.formula import parse_dimacs_text
from tensororder_amd.instances import random_3cnf


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
