"""The executor's work as its users have it done, for timing.

A case is one pass through a public entry point: a whole count of one formula on a plan that
the program keeps (``HipAPI.prepare``), a batch of formulas (``prepare_batch``), the plugin
call ``contract_sliced`` that compiles and runs a plan, one join (``HipAPI.tensordot`` and the
C entry ``to_tensordot``), and one training step of the plan-cost model.  Plans come from the
committed fixtures (tests/golden) or from the package's own planners on seeded random
formulas of the benchmark's two families: weighted vertex cover of 3-regular graphs (line
plans) and weighted random 3-CNF (factor plans, sliced).  A seed gives the literal weights
w(x) ~ U(0.1, 0.9) of a count, or the entries of a join's tensors, or a training batch.
"""

import ctypes
import functools
import json
import math
import os
import random

import numpy as np
import torch

from tensororder_amd import _lib, costmodel, decomposition, network, plan_io, planners
from tensororder_amd.formula import parse_dimacs_text
from tensororder_amd.hip_api import DeviceTensor, HipAPI, HipF32API
from tensororder_amd.instances import random_3cnf, vertex_cover_cnf
from tensororder_amd.plan import ALL_SLICERS

GOLDEN = os.path.join("tests", "golden")
# device memory one executor may use: several plans stay resident on one card
MEM_LIMIT = 72 << 30


def listed():
    return [
        # the smallest counts: a program that counts many small formulas one after another
        # waits for launches, not for arithmetic
        {"name": "count_vc24_f64", "kind": "count", "source": "vc24_weighted_factor_s5", "f32": False},
        # ordinary counts, one formula at a time, in both entry types
        {"name": "count_vc60_f32", "kind": "count", "source": "vc", "n": 60, "id": 1, "f32": True},
        {"name": "count_vc90_f64", "kind": "count", "source": "vc90_weighted_line", "f32": False},
        {"name": "count_cnf40_f64", "kind": "count", "source": "cnf40_factor_s6", "f32": False},
        # the benchmark's large line plan: rank 28, one product of 2^39 multiply-adds
        {"name": "count_vc200_f32", "kind": "count", "source": "vc200_weighted_line", "f32": True},
        # the benchmark's headline: 4096 slices of a 70-variable formula on the plan that the
        # learned model picks; the plain FP64 executor on the first slices of the reference
        # rule's plan (slice prefixes are the reference's --slice_cutoff)
        {"name": "count_cnf70_f32", "kind": "count", "source": "cnf70_candidate", "f32": True},
        {"name": "count_cnf70_64s_f64", "kind": "count", "source": "cnf70_factor_s12", "limit": 64, "f32": False},
        # many formulas at once: the mixed batch's first instances
        {"name": "batch96_f32", "kind": "batch", "source": "vc_batch512", "count": 96, "f32": True},
        # the plugin call as execution.run makes it: compile the plan, upload, contract
        {"name": "call_cnf20_f64", "kind": "call", "source": "cnf20_factor_s4", "f32": False},
        # one join through the plugin: a dense product in the FP32-scaled executor
        {"name": "tensordot_dense_f32", "kind": "tensordot", "ra": 23, "rb": 21, "s": 10, "id": 3, "f32": True},
        # one join through the C entry point: a large tensor absorbs a small one
        {"name": "c_tensordot_absorb_f64", "kind": "c_tensordot", "ra": 23, "rb": 6, "s": 3, "id": 4, "f32": False},
        # one step of the plan-cost model's training loop (forward, backward, Adam)
        {"name": "train_2048", "kind": "train", "rows": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["count", "count", "count", "count", "batch", "call", "tensordot", "c_tensordot", "train"])
    f32 = rng.random() < 0.5
    ident = rng.randrange(1 << 20)
    if kind in ("count", "call"):
        if rng.random() < 0.5:
            n = 2 * rng.randint(8, 55 if kind == "count" else 30)
            return {"kind": kind, "source": "vc", "n": n, "id": ident, "f32": f32}
        n = rng.randint(16, 50 if kind == "count" else 30)
        return {"kind": kind, "source": "cnf", "n": n, "m": int(round(n * rng.uniform(1.6, 2.2))),
                "slices": rng.randint(0, 7), "id": ident, "f32": f32}
    if kind == "batch":
        return {"kind": kind, "source": "vc", "count": _log_int(rng, 3, 48), "low": 2 * rng.randint(8, 20),
                "high": 2 * rng.randint(22, 40), "id": ident, "f32": f32}
    if kind == "train":
        return {"kind": kind, "rows": _log_int(rng, 200, 8192)}
    # joins from small to large: outputs of at most 2^24 entries, at most 2^33 products
    while True:
        s = rng.randint(0, 12)
        fx, fy = rng.randint(2, 20), rng.randint(0, 12)
        if fy <= fx and fx + fy <= 24 and fx + s <= 24 and 12 <= fx + fy + s <= (33 if kind == "tensordot" else 27):
            break
    if rng.random() < 0.5:
        fx, fy = fy, fx
    return {"kind": kind, "ra": fx + s, "rb": fy + s, "s": s, "id": ident, "f32": f32}


# ---------------------------------------------------------------------------------------
# formulas and plans


def _weights(text):
    """{variable: weight} of the ``w`` lines of a DIMACS text."""
    return {int(l.split()[1]): float(l.split()[2]) for l in text.splitlines() if l.startswith("w ")}


@functools.lru_cache(maxsize=None)
def _golden(name):
    with open(os.path.join(GOLDEN, name + ".json")) as f:
        return json.load(f)


@functools.lru_cache(maxsize=64)
def _template(source, n=0, m=0, slices=0, ident=0):
    """(DIMACS text, plan document) of one formula with its own weights."""
    if source == "cnf70_candidate":
        # the 70-variable formula's candidate that the learned model picks: the greedy_largest
        # slices with random seed 1 of the third decomposition
        doc = _golden("cnf70_candidates")
        net = network.cnf_count(parse_dimacs_text(doc["dimacs"], doc["weights"]))
        td = decomposition.parse_all(doc["decompositions"][2]["text"])[0]
        plans, labels = planners.plan_candidates(net, "factor", [td], doc["slices"])
        pick = [p for p, lab in zip(plans, labels) if lab["slicer"] == "greedy_largest" and lab["seed"] == 1]
        return doc["dimacs"], plan_io.plan_to_dict(pick[0])
    if source == "vc" or source == "cnf":
        text = vertex_cover_cnf(n, ident, True) if source == "vc" else random_3cnf(n, m, ident, True)
        net = network.cnf_count(parse_dimacs_text(text, "cachet"))
        plan = planners.best_plan(net, "line" if source == "vc" else "factor", solver=None, seed=0)
        state = random.getstate()
        random.seed(0)
        try:
            ALL_SLICERS["greedy_mem"].slice_until(plan, rank=24, slices=slices)
        finally:
            random.setstate(state)
        return text, plan_io.plan_to_dict(plan)
    doc = _golden(source)
    return doc["meta"]["dimacs"], doc


@functools.lru_cache(maxsize=1)
def _batch_templates():
    doc = _golden("vc_batch512")
    plans, _ = plan_io.batch_plans(dict(doc, instances=doc["instances"][:96]))
    return [(vertex_cover_cnf(row["n"], row["seed"], True), plan_io.plan_to_dict(p))
            for row, p in zip(doc["instances"], plans)]


def _templates(case):
    """The (text, plan document) pairs of a case, one per formula."""
    if case["kind"] != "batch":
        return [_template(case["source"], case.get("n", 0), case.get("m", 0), case.get("slices", 0), case.get("id", 0))]
    if case["source"] == "vc_batch512":
        return _batch_templates()[:case["count"]]
    rng = random.Random(case["id"])
    return [_template("vc", 2 * rng.randint(case["low"] // 2, case["high"] // 2), 0, 0, rng.randrange(1 << 20))
            for _ in range(case["count"])]


def _reweighted(text, seed, which):
    """{variable: new weight w(x)} of formula number ``which``."""
    rng = np.random.default_rng([seed, which])
    return {v: float(p) for v, p in zip(sorted(_weights(text)), rng.uniform(0.1, 0.9, len(_weights(text))))}


def _plan(text, doc, new):
    """The plan with its formula's weights replaced."""
    by_old = {p: new[v] for v, p in _weights(text).items()}
    tensors = [dict(t, w_pos=by_old[t["w_pos"]], w_neg=1 - by_old[t["w_pos"]])
               if t["kind"] == "var" and t["w_pos"] in by_old else t for t in doc["tensors"]]
    return plan_io.plan_from_dict(dict(doc, tensors=tensors))


def _plans(case, seed):
    return [_plan(text, doc, _reweighted(text, seed, i)) for i, (text, doc) in enumerate(_templates(case))]


# ---------------------------------------------------------------------------------------
# inputs of the joins and of the training step


def _axes(case):
    rng = random.Random(case["id"])
    return (sorted(rng.sample(range(case["ra"]), case["s"])), rng.sample(range(case["rb"]), case["s"]))


def _operands(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = torch.float32 if case["f32"] else torch.float64
    return tuple(torch.rand(1 << r, dtype=dt, device="cuda", generator=gen) for r in (case["ra"], case["rb"]))


def _record():
    """A scale record of a tensor stored with exponent 0 and entries below 1."""
    return torch.tensor([0, int(np.float32(1.0).view(np.uint32))], dtype=torch.int64, device="cuda")


def _rows(case, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((case["rows"], 16)).astype(np.float32)
    t = np.tanh(x @ rng.standard_normal((16, 2)).astype(np.float32)) + 0.1 * rng.standard_normal((case["rows"], 2))
    return x, t.astype(np.float32)


# ---------------------------------------------------------------------------------------
# the passes


class _State:
    def __init__(self, **kw):
        self.exe = None
        self.__dict__.update(kw)

    def __del__(self):
        if self.exe is not None:
            self.exe.close()


def prepare(case, seed):
    api = HipF32API() if case.get("f32") else HipAPI()
    api.add_argument("mem_limit", MEM_LIMIT)
    kind = case["kind"]
    if kind == "count":
        return _State(case=case, exe=api.prepare(_plans(case, seed)[0], case.get("limit")))
    if kind == "batch":
        return _State(case=case, exe=api.prepare_batch(_plans(case, seed)))
    if kind == "call":
        return _State(case=case, api=api, plan=_plans(case, seed)[0])
    if kind == "train":
        x, t = _rows(case, seed)
        return _State(case=case, model=costmodel.CostModel(api, seed=seed), x=torch.from_numpy(x).cuda(),
                      t=torch.from_numpy(t).cuda())
    a, b = _operands(case, seed)
    recs = [_record() for _ in range(3)] if case["f32"] else [None] * 3
    if kind == "tensordot":
        A, B = (DeviceTensor(t, (2,) * r, None if rec is None else rec.view(torch.uint8), api)
                for t, r, rec in zip((a, b), (case["ra"], case["rb"]), recs))
        torch.cuda.synchronize()
        return _State(case=case, api=api, A=A, B=B, axes=_axes(case))
    la, lb = ((ctypes.c_int32 * max(1, case["s"]))(*v) for v in _axes(case))
    lib, et = _lib.load(), _lib.TO_F32S if case["f32"] else _lib.TO_F64
    need = ctypes.c_int64()
    _lib.check(lib.to_tensordot_workspace(case["ra"], case["rb"], ctypes.addressof(la), ctypes.addressof(lb),
                                          case["s"], et, ctypes.byref(need)), "to_tensordot_workspace")
    return _State(case=case, lib=lib, a=a, b=b, recs=recs, la=la, lb=lb, et=et,
                  c=torch.empty(1 << (case["ra"] + case["rb"] - 2 * case["s"]), dtype=a.dtype, device="cuda"),
                  work=torch.empty(max(8, need.value), dtype=torch.uint8, device="cuda"), need=need.value)


def _numbers(mants, exps, f32):
    """Counts as (mantissa in [0.5, 1), exponent), the mantissas in the executor's precision
    (counts of large formulas leave float32's range)."""
    pairs = [math.frexp(m) for m in mants]
    return {"mantissa": np.array([m for m, _ in pairs], dtype=np.float32 if f32 else np.float64),
            "exponent": np.array([e + x for (_, e), x in zip(pairs, exps)], dtype=np.int64)}


def run(state):
    case = state.case
    kind = case["kind"]
    if kind == "count":
        r = state.exe.run()
        return _numbers([r.mant], [r.exp], case["f32"])
    if kind == "batch":
        res, _ = state.exe.run()
        return _numbers([r.mant for r in res], [r.exp for r in res], case["f32"])
    if kind == "call":
        return _numbers([state.api.contract_sliced(state.plan)], [0], case["f32"])
    if kind == "train":
        loss, grad = state.model.gradient(state.x, state.t)
        state.model.adam_step()
        return {"loss": loss, "grad": grad, "params": state.model.params}
    if kind == "tensordot":
        out = state.api.tensordot(state.A, state.B, state.axes)
        if not case["f32"]:
            return {"data": out.data}
        return {"data": out.data, "exponent": out.rec[:8].view(torch.int64)}
    p = ctypes.c_void_p
    recs = [p(r.data_ptr()) if r is not None else None for r in state.recs]
    _lib.check(state.lib.to_tensordot(p(state.a.data_ptr()), p(state.b.data_ptr()), p(state.c.data_ptr()),
                                      case["ra"], case["rb"], ctypes.addressof(state.la), ctypes.addressof(state.lb),
                                      case["s"], state.et, recs[0], recs[1], recs[2], p(state.work.data_ptr()),
                                      state.need, p(torch.cuda.current_stream().cuda_stream)), "to_tensordot")
    if not case["f32"]:
        return {"data": state.c}
    return {"data": state.c, "exponent": state.recs[2][:1]}


# ---------------------------------------------------------------------------------------
# what a pass cannot do without, and its results in 64 bits


@functools.lru_cache(maxsize=256)
def _plan_products(source, n, m, slices, ident, which=None):
    """(multiply-adds of one slice, leaf entries, slices) of a plan: a join costs one
    product per assignment of the distinct variables (and OR-gate wires) it touches -- the
    edges that COPY tensors force equal counted once."""
    doc = (_batch_templates()[which] if which is not None else _template(source, n, m, slices, ident))[1]
    root = list(range(len(doc["edges"])))

    def find(e):
        while root[e] != e:
            e = root[e]
        return e

    for t, edges in zip(doc["tensors"], doc["index_lists"]):
        if t["kind"] == "var":
            for e in edges[1:]:
                root[find(e)] = find(edges[0])
    cut = {find(e) for g in doc["groups_to_slice"] for e in g}
    stack, products, entries = [], 0, 0
    for tok in doc["tree"]:
        if tok >= 0:
            edges = set(doc["index_lists"][tok])
            entries += 1 << len({find(e) for e in edges})
        else:
            right, left = stack.pop(), stack.pop()
            products += 1 << len({find(e) for e in left | right} - cut)
            edges = left ^ right
        stack.append(edges)
    return products, entries, 1 << sum(1 for g in doc["groups_to_slice"] if g)


def work(case):
    e = 4 if case.get("f32") else 8
    if case["kind"] in ("count", "call", "batch"):
        if case["kind"] == "batch" and case["source"] == "vc_batch512":
            args = [(case["source"], 0, 0, 0, 0, i) for i in range(case["count"])]
        elif case["kind"] == "batch":
            rng = random.Random(case["id"])
            args = [("vc", 2 * rng.randint(case["low"] // 2, case["high"] // 2), 0, 0, rng.randrange(1 << 20))
                    for _ in range(case["count"])]
        else:
            args = [(case["source"], case.get("n", 0), case.get("m", 0), case.get("slices", 0), case.get("id", 0))]
        flops = nbytes = 0
        for a in args:
            products, entries, slices = _plan_products(*a)
            flops += 2 * products * min(slices, case.get("limit", slices))
            nbytes += entries * e + 16
        return {"bytes": nbytes, "flops": flops}
    if case["kind"] == "train":
        params = 16 * 64 + 64 + 64 * 64 + 64 + 64 * 2 + 2
        # forward, activation gradients, weight gradients; inputs and targets read, the
        # parameters and both moments read and written, the gradient written
        return {"bytes": 4 * (case["rows"] * 18 + 7 * params), "flops": 6 * case["rows"] * params}
    out = case["ra"] + case["rb"] - 2 * case["s"]
    return {"bytes": e * ((1 << case["ra"]) + (1 << case["rb"]) + (1 << out)), "flops": 2 << (out + case["s"])}


def _count(text, weights, limit=26):
    """The weighted count of a CNF by eliminating its variables one at a time (the variable
    whose elimination makes the smallest table first), in float64; None where a table would
    exceed 2^limit entries."""
    clauses = [[int(x) for x in l.split()[:-1]] for l in text.splitlines() if l and l[0] not in "pwc"]
    tables = []
    for c in clauses:
        vs = sorted(abs(x) for x in c)
        t = np.ones((2,) * len(vs))
        t[tuple(0 if v in c else 1 for v in vs)] = 0.0
        tables.append((vs, t))
    total, left = 1.0, set(weights)
    while left:
        def size(v):
            return len(set().union(*[set(vs) for vs, _ in tables if v in vs] or [set()]))

        v = min(sorted(left), key=size)
        if size(v) > limit:
            return None
        left.remove(v)
        mine = [x for x in tables if v in x[0]]
        tables = [x for x in tables if v not in x[0]]
        w = np.array([1.0 - weights[v], weights[v]])
        if not mine:
            total *= float(w.sum())
            continue
        vs = [v] + sorted(set().union(*[set(x[0]) for x in mine]) - {v})
        acc = w.reshape([2] + [1] * (len(vs) - 1))
        for names, t in mine:
            order = sorted(range(len(names)), key=lambda i: vs.index(names[i]))
            shape = [2 if u in names else 1 for u in vs]
            acc = acc * np.transpose(t, order).reshape(shape)
        acc = np.broadcast_to(acc, (2,) * len(vs)).sum(axis=0)
        if vs[1:]:
            tables.append((vs[1:], acc))
        else:
            total *= float(acc)
    return total


def exact(case, seed):
    kind = case["kind"]
    if kind in ("count", "call", "batch"):
        if case.get("limit") or case["source"] in ("vc200_weighted_line", "cnf70_candidate", "vc_batch512"):
            return None  # a slice prefix, or tables that take a host too long
        counts = [_count(text, _reweighted(text, seed, i)) for i, (text, _) in enumerate(_templates(case))]
        if any(c is None for c in counts):
            return None
        return _numbers(counts, [0] * len(counts), False)
    if kind == "train":
        return _train_step(case, seed)
    a, b = (t.cpu().double().numpy().reshape((2,) * r) for t, r in zip(_operands(case, seed), (case["ra"], case["rb"])))
    la, lb = _axes(case)
    fa, fb = ([i for i in range(r) if i not in l] for r, l in ((case["ra"], la), (case["rb"], lb)))
    left = np.ascontiguousarray(a.transpose(fa + list(la))).reshape(1 << len(fa), 1 << case["s"])
    right = np.ascontiguousarray(b.transpose(list(lb) + fb)).reshape(1 << case["s"], 1 << len(fb))
    out = (torch.from_numpy(left).cuda() @ torch.from_numpy(right).cuda()).reshape(-1)
    # the scaled executor stores the result of two tensors recorded with max 1.0 as 2^-2 of it
    return {"data": out / 4, "exponent": None} if case["f32"] else {"data": out}


def _train_step(case, seed):
    x, t = (v.astype(np.float64) for v in _rows(case, seed))
    rng = np.random.default_rng(seed)  # the model's own initial parameters for this seed
    W, B = [], []
    for dout, din in ((64, 16), (64, 64), (2, 64)):
        W.append((rng.standard_normal((dout, din)) * math.sqrt(2.0 / din)).astype(np.float32).astype(np.float64))
        B.append(np.zeros(dout))
    h1 = np.maximum(x @ W[0].T + B[0], 0.0)
    h2 = np.maximum(h1 @ W[1].T + B[1], 0.0)
    y = h2 @ W[2].T + B[2]
    dy = 2.0 * (y - t) / y.size
    d2 = (dy @ W[2]) * (h2 > 0)
    d1 = (d2 @ W[1]) * (h1 > 0)
    grad = np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), (dy.T @ h2).ravel(), dy.sum(0)])
    # one bias-corrected Adam step from zero moments moves each parameter by lr g / (|g| + eps)
    p = np.concatenate([v.ravel() for pair in zip(W, B) for v in pair])
    return {"loss": np.float64(np.mean((y - t) ** 2)), "grad": grad, "params": p - 3e-3 * grad / (np.abs(grad) + 1e-8)}
