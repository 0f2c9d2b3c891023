"""Runs of an executable that do not go their usual way: cut short while they are queued, or their
launches run by a caller."""

import json
import os

import pytest
from emulated import EmulatedAPI

from oracle import numpy_oracle
from tensororder_amd import _lib, hip_api, plan_io

PLAN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "cnf20_factor_s4.json")


def _plan():
    with open(PLAN) as f:
        plan = plan_io.plan_from_dict(json.load(f))
    return plan, numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))


@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_runs_after_one_cut_short(et, tol):
    plan, want = _plan()
    api = EmulatedAPI(et, max_batch=4)
    exe = api.prepare(plan)
    launches = sum(len(run) for _, run in exe._runs)
    assert exe.nwaves == 4 and launches > 8
    for before in (0, 1):  # runs queued before the one cut short
        for k in range(launches):
            for _ in range(before):
                exe.enqueue()
            api.fail_at = k
            with pytest.raises(KeyboardInterrupt):
                exe.run()
            with pytest.raises(RuntimeError):
                exe.result()
            for _ in range(2):
                r = exe.run()
                assert r.value == pytest.approx(want, rel=tol) and r.slices == exe.total
    waits = api.waits
    api.fail_at = 2
    with pytest.raises(KeyboardInterrupt):
        exe.enqueue()
    exe.close()
    assert api.waits == waits + 1  # launches of the cut run may still write its memory
    assert exe.run().value == pytest.approx(want, rel=tol)


@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_runs_between_launches_of_a_caller(et, tol):
    plan, want = _plan()
    api = EmulatedAPI(et, max_batch=4)
    exe = api.prepare(plan)
    assert exe.run().value == pytest.approx(want, rel=tol)
    step, wave = exe.step_launches, exe.wave_launches
    for run in (step, wave, step + wave, step + wave * 3):
        api._run(run)
        r = exe.run()
        assert r.value == pytest.approx(want, rel=tol) and r.slices == exe.total
    api._run(step + wave * 4)
    assert exe.result().value == pytest.approx(want, rel=tol)


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [True, False])
def test_runs_after_one_cut_short_on_the_device(graph, monkeypatch):
    plan, want = _plan()
    monkeypatch.setattr(hip_api.Executable, "ONE_GRAPH_LAUNCHES", 1)
    api = hip_api.HipAPI()
    api.add_argument("graph", graph)
    api.add_argument("max_batch", 4)
    exe = api.prepare(plan)
    name = "_launch_graph" if graph else "_run"
    where = exe if graph else api
    inner = getattr(where, name)
    for k in range(5):
        calls = iter(range(100))

        def cut(run):
            if next(calls) == k:
                raise KeyboardInterrupt
            inner(run)

        print("case run cut short", graph, k, flush=True)
        setattr(where, name, cut)
        with pytest.raises(KeyboardInterrupt):
            exe.run()
        setattr(where, name, inner)
        with pytest.raises(RuntimeError):
            exe.result()
        for _ in range(3):
            r = exe.run()
            assert r.value == pytest.approx(want, rel=1e-12) and r.slices == exe.total
    exe.close()
