"""The edge-by-edge executor on the device: plans with COPY leaves are folded, so the tests of
counts and batches are repeated here with folding switched off."""

import json
import os

import pytest
import test_gpu_parity as parity
from test_gpu_parity import hip, hip32  # noqa: F401 (fixtures)

from tensororder_amd import _lib, fold, plan_io

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def walk(monkeypatch):
    monkeypatch.setattr(fold, "has_copies", lambda tables: False)


PLANS = [p for p in parity.FULL if parity._name(p) in ("cnf20_factor_s4", "vc24_weighted_factor_s5", "vc22_weighted_line_s3",
                                                       "vc90_weighted_line", "cnf40_factor_s6")]


@pytest.mark.parametrize("path", PLANS, ids=[parity._name(p) for p in PLANS])
def test_counts(hip, hip32, path):  # noqa: F811
    parity.test_fixture_fp64(hip, path)
    parity.test_fixture_fp32_scaled(hip32, path)


def test_batch_sizes(hip):  # noqa: F811
    parity.test_batch_sizes_and_prefix(hip, 3)
    parity.test_graph_and_eager_agree(hip)


def test_uneven_batch(hip, hip32):  # noqa: F811
    parity.test_batch_of_uneven_instances(hip, hip32)


def test_batch_of_the_fixture(hip, hip32):  # noqa: F811
    # grouped launches of mixed streamed joins, of one-wave joins, and block maps are among them
    with open(os.path.join(parity.HERE, "golden", "vc_batch512.json")) as f:
        doc = json.load(f)
    plans, wants = plan_io.batch_plans(dict(doc, instances=doc["instances"][:48]))
    print("case edge walk, batch of", len(plans), flush=True)
    for api, tol in ((hip, parity.F64_TOL), (hip32, parity.F32_TOL)):
        exe = api.prepare_batch(plans)
        launches = [L for prog in exe.progs for L in prog.launches]
        streams = {L.variant for L in launches if L.op == _lib.TO_OP_JOIN_STREAM}
        assert streams == {_lib.TO_STREAM_ANY, _lib.TO_STREAM_WAVE} and any(L.aux1 for L in launches)
        for _ in range(3):
            res, _lat = exe.run()
            assert [r.value for r in res] == pytest.approx(wants[:len(plans)], rel=tol)
        exe.close()
