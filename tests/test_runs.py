"""Runs of an executable that do not go their usual way: cut short while they are queued, or their
launches run by a caller, or that never come."""

import json
import os

import numpy as np
import pytest
from emulated import EmulatedAPI

from oracle import numpy_oracle
from tensororder_amd import _lib, hip_api, plan_io

PLAN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "cnf20_factor_s4.json")


def _plan():
    with open(PLAN) as f:
        plan = plan_io.plan_from_dict(json.load(f))
    return plan, numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))


def _unsliced():
    with open(PLAN) as f:
        return plan_io.plan_from_dict(dict(json.load(f), groups_to_slice=[]))


@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_runs_after_one_cut_short(et, tol):
    plan, want = _plan()
    api = EmulatedAPI(et, max_batch=4)
    exe = api.prepare(plan)
    launches = sum(len(run) for _, run in exe._runs)
    assert exe.nwaves == 4 and launches > 8
    for k in range(0, launches, 3):
        if k % 2:  # a run is queued before the one cut short
            exe.enqueue()
        api.fail_at = k
        with pytest.raises(KeyboardInterrupt):
            exe.run()
        with pytest.raises(RuntimeError):
            exe.result()
        for _ in range(1 + (k % 4 == 0)):
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


def test_runs_of_no_slices():
    # no sum ends such a run: its prologue is waited for
    plan, _ = _plan()
    api = EmulatedAPI()
    exe = api.prepare(plan, 0)
    assert exe.nwaves == 0 and exe.run().value == 0.0 and api.waits == 1


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


@pytest.mark.parametrize("make", ["prepare", "prepare_batch"])
def test_dropped_before_the_first_run(make):
    # small uploads are queued, not waited for: the memory they write is not given back before
    plan, want = _plan()
    plans = plan if make == "prepare" else [_unsliced()]
    for how in ("drop", "close", "run"):
        api = EmulatedAPI(_lib.TO_F32S)
        exe = getattr(api, make)(plans)
        assert api.waits == 0
        if how == "close":
            exe.close()
            assert api.waits == 1
        if how == "run":
            exe.run()
        waits = api.waits
        del exe
        assert api.waits == waits + (how == "drop")
    # ... nor where making it resident fails half-way
    api = EmulatedAPI(_lib.TO_F32S)
    for k in range(1, 3):
        done = []

        def upload(dst, data):
            if len(done) == k:
                raise hip_api.OutOfMemoryError
            done.append(dst)

        api._upload = upload
        waits = api.waits
        with pytest.raises(hip_api.OutOfMemoryError):
            getattr(api, make)(plans)
        assert api.waits == waits + 1
        del api._upload


def test_failed_joins_wait_for_their_operands():
    api, sent = EmulatedAPI(), []
    api._to_device = lambda t: sent.append(t) or t
    with pytest.raises(ValueError):  # refused before anything is sent
        api.tensordot(np.ones((2, 2)), np.ones((2, 3)), ([0], [0]))
    assert not sent and not api.waits

    def fail(*args):
        raise hip_api.OutOfMemoryError

    api._tensordot = api._permute = fail
    with pytest.raises(hip_api.OutOfMemoryError):
        api.tensordot(np.ones((2, 2)), np.ones((2, 2)), ([0], [0]))
    with pytest.raises(hip_api.OutOfMemoryError):
        api.permute(np.ones((2, 2)), (1, 0))
    assert len(sent) == 3 and api.waits == 2


@pytest.mark.gpu
@pytest.mark.parametrize("make", ["prepare", "prepare_batch"])
def test_dropped_before_the_first_run_on_the_device(make):
    import torch

    api = hip_api.HipF32API()
    plan, _ = _plan()
    busy = api.prepare(plan)
    for k in range(5):
        print("case dropped before its run", make, k, flush=True)
        for _ in range(50):
            busy.enqueue()
        exe = getattr(api, make)(plan if make == "prepare" else [_unsliced()])
        del exe
        # memory of the sizes it had, on the caller's stream
        fresh = [torch.full((n,), 7, dtype=torch.uint8, device="cuda") for n in (16, 32, 512, 4096, 65536, 1 << 20) * 8]
        torch.cuda.synchronize()
        api.synchronize()
        assert all(bool((t == 7).all()) for t in fresh)
    busy.result()
    busy.close()
