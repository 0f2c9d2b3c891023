"""Folded plans (COPY tensors as index identities): the compiled records, executed by a numpy
emulator of to_fold_desc, reproduce the oracle over plans, slicings, entry types and batch
sizes; the kernels match float64 sums over every form, on the GPU."""

import ctypes
import json
import math
import os
import types

import numpy as np
import pytest
from fixtures import plan_fixture_paths

import emulator
from oracle import numpy_oracle
from tensororder_amd import _lib, fold, hip_api, network, plan_io, planners, schedule
from tensororder_amd.formula import parse_dimacs_text
from tensororder_amd.instances import random_3cnf, vertex_cover_cnf
from tensororder_amd.plan import ALL_SLICERS

HERE = os.path.dirname(os.path.abspath(__file__))
SMALL = [f for f in plan_fixture_paths() if json.load(open(f))["meta"]["maxrank"] <= 16]


def _say(*args):
    print(*args, flush=True)


def _spread(entries, lo, n):
    """What each value of bits [lo, lo + n) of a descriptor adds to an offset."""
    out = np.zeros(1, dtype=np.int64)
    for i in range(lo, lo + n):
        out = np.concatenate([out, out + int(entries[i])])
    return out


class FoldEmulator(emulator.Emulator):
    TABLE_DESCS = {**emulator.Emulator.TABLE_DESCS, _lib.TO_OP_FOLD: "FoldDesc", _lib.TO_OP_FOLD_TREE: "TreeDesc",
                   _lib.TO_OP_FOLD_PAIR: "PairDesc"}

    def __init__(self, heap, entry_type):
        super().__init__(heap, entry_type)
        self.forms = set()

    def op_16(self, L):
        # leaf gather and record clearing in one launch: whatever the order, neither touches
        # what the other writes
        gathered = [self.heap.read_struct(_lib.LeafDesc, L.descs + i * ctypes.sizeof(_lib.LeafDesc))
                    for i in range(L.count)]
        assert sum(d.nblocks for d in gathered) == L.iaux1 <= L.grid
        for d in gathered:
            assert not L.iaux0 or d.rec + 16 * d.nbatch <= L.aux0 or d.rec >= L.aux0 + 16 * L.iaux0
        self.op_1(L)
        if L.iaux0:
            assert L.grid > L.iaux1
            self.op_5(L)

    def op_6(self, L):
        assert L.variant == 1
        params = self.heap.view(L.aux3, np.int64, 2)
        if params[0] == 0:
            off = L.aux2 - emulator.HEAP_BASE
            self.heap.mem[off:off + ctypes.sizeof(_lib.Accum)] = 0
        super().op_6(L)
        params[0] = params[0] + L.iaux0 if params[0] + L.iaux0 < params[1] else 0
        acc = bytes(self.heap.read_struct(_lib.Accum, L.aux2))
        if L.iaux1:
            off = L.iaux1 - emulator.HEAP_BASE
            self.heap.mem[off:off + len(acc)] = np.frombuffer(acc, np.uint8)

    def op_14(self, L):
        size = ctypes.sizeof(_lib.FoldDesc)
        for i in range(L.count):
            d = self.heap.read_struct(_lib.FoldDesc, L.descs + i * size)
            vec = L.variant & _lib.TO_FOLD_VEC
            self.forms.add(L.variant)
            if vec:
                assert d.nreg == (L.variant & 15) and d.lo == 10 and d.lk == 0 and d.lsplit == 0
                assert list(d.bx[:2]) == [1, 2] and list(d.bc[:2]) == [1, 2]
                ym = {(0, 0): 0, (1, 2): 1}.get(tuple(d.by[:2]), 2 if d.by[0] and d.by[1] else 3 if d.by[0] else 4)
                at = 10 + d.ntile + d.nloop
                ym = 5 if not ym and d.nreg >= 2 and list(d.by[at:at + 2]) == [1, 2] else ym
                # (the batch runs modes 3 to 5 in the general ones)
                assert (L.variant >> 4) & 15 in (ym, {3: 2, 4: 2, 5: 0}.get(ym, ym))
                ym = (L.variant >> 4) & 15
                # 4-element alignment of everything the 16-byte form loads or stores at once
                for ptr, stride, arr, used, low in ((d.x, d.xb, d.bx, True, 0), (d.c, d.cb, d.bc, True, 0),
                                                    (d.y, d.yb, d.by, ym in (1, 5), at if ym == 5 else 0)):
                    if used:
                        assert ptr % (4 * self.dt().itemsize) == 0 and stride % 4 == 0
                        assert all(int(e) % 4 == 0 for i, e in enumerate(arr) if not low <= i < low + 2)
                thr, tile0 = (0, 10), 10
            elif L.variant & _lib.TO_FOLD_REG:
                na, nb = L.variant >> 4 & 15, L.variant & 15
                assert d.nreg == na + nb and d.lo == 8 and d.lk == 0 and d.lsplit == 0
                r0 = 8 + d.ntile + d.nloop
                assert not any(list(d.by)[r0:r0 + na]) and not any(list(d.bx)[r0 + na:r0 + d.nreg])
                thr, tile0 = (0, 8), 8
            else:
                assert d.nreg == 0 and d.lo + d.lk <= 8 and all(int(e) == 0 for e in list(d.bc)[d.lo:8])
                thr, tile0 = (0, d.lo), 8
            k0 = tile0 + d.ntile
            r0 = k0 + d.nloop + d.lsplit
            assert r0 + d.nreg <= _lib.FOLD_BITS
            offs = []
            bx, by, bc = list(d.bx), list(d.by), list(d.bc)
            for arr in (bx, by, bc):
                o = (_spread(arr, *thr)[None, None, :] + _spread(arr, tile0, d.ntile)[None, :, None]
                     + _spread(arr, r0, d.nreg)[:, None, None]).ravel()
                k = (_spread(arr, d.lo, 0 if vec else d.lk)[None, :]
                     + _spread(arr, k0, d.nloop + d.lsplit)[:, None]).ravel()
                if L.variant == _lib.TO_FOLD_DOT:
                    four = np.arange(4) if arr is not bc else np.zeros(4, dtype=np.int64)
                    if arr is not bc:
                        assert all(int(e) % 4 == 0 for e in arr) and d.x % 16 == d.y % 16 == 0
                        assert d.xb % 4 == d.yb % 4 == 0
                    k = (k[:, None] + four[None, :]).ravel()
                offs.append((o, k))
            co = offs[2][0]
            assert np.array_equal(np.sort(co), np.arange(co.size))  # every output once
            assert not np.any(offs[2][1])
            esz = self.dt().itemsize
            for b in range(d.nbatch):
                xo = offs[0][0][:, None] + offs[0][1][None, :]
                yo = offs[1][0][:, None] + offs[1][1][None, :]
                X = self.heap.view(d.x + b * d.xb * esz, self.dt, int(xo.max()) + 1).astype(np.float64)
                Y = self.heap.view(d.y + b * d.yb * esz, self.dt, int(yo.max()) + 1).astype(np.float64)
                e = 0
                f = 1.0
                if self.scaled:
                    for rec in (self.get_rec(d.xs, b * d.xsb), self.get_rec(d.ys, b * d.ysb)):
                        e += rec[0] + emulator._scale_exp(rec[1])
                        f *= 2.0 ** -emulator._scale_exp(rec[1])
                prod = X[xo] * Y[yo]
                if d.lsplit:
                    S = 1 << d.lsplit
                    P = self.heap.view(d.partial, np.float64, (d.nbatch * co.size) << d.lsplit)
                    # shared index = (split, loop, thread bits)
                    parts = prod.reshape(co.size, S, -1).sum(axis=2) * f
                    for sp in range(S):
                        P[((b * co.size + co) << d.lsplit) | sp] = parts[:, sp]
                    self.gemm_partials.add(d.partial)
                    continue
                val = (prod.sum(axis=1) * f).astype(self.dt)
                self.heap.view(d.c + b * d.cb * esz, self.dt, co.size)[co] = val
                if self.scaled:
                    m = np.float32(np.max(np.abs(val)))
                    self.set_rec(d.cs, b, exp=e, maxbits=int(m.view(np.uint32)))

    def op_17(self, L):
        esz = self.dt().itemsize
        for i in range(L.count):
            d = self.heap.read_struct(_lib.PairDesc, L.descs + i * ctypes.sizeof(_lib.PairDesc))
            self.forms.add((_lib.TO_OP_FOLD_PAIR, L.variant))
            one = 0 if any(list(d.by[0])[:2] + list(d.by[1])[:2]) else _lib.TO_PAIR_ONE
            assert L.variant == d.nk[0] << 4 | d.nk[1] | one and d.nk[0] >= d.nk[1]
            ka = 10 + d.nloop + d.lsplit + d.nreg
            assert ka + sum(d.nk) <= _lib.FOLD_BITS and not any(list(d.bx[0])[ka - d.nreg:ka])
            for b in range(d.nbatch):
                side, f, exps = [], 1.0, []
                for k in range(2):
                    bx, by = list(d.bx[k]), list(d.by[k])
                    assert bx[:2] == [1, 2] and all(int(e) % 4 == 0 for e in bx[2:])
                    assert d.x[k] % (4 * esz) == 0 and d.xb[k] % 4 == 0
                    first = ka + (d.nk[0] if k else 0)
                    xo, yo = (_spread(arr, 0, ka)[:, None] + _spread(arr, first, d.nk[k])[None, :] for arr in (bx, by))
                    X = self.heap.view(d.x[k] + b * d.xb[k] * esz, self.dt, int(xo.max()) + 1).astype(np.float64)
                    Y = self.heap.view(d.y[k] + b * d.yb[k] * esz, self.dt, int(yo.max()) + 1).astype(np.float64)
                    side.append((X[xo] * Y[yo]).sum(axis=1))
                    if self.scaled:
                        recs = [self.get_rec(at, b * stride)
                                for at, stride in ((d.xs[k], d.xsb[k]), (d.ys[k], d.ysb[k])) if at]
                        exps.append(sum(r[0] + emulator._scale_exp(r[1]) for r in recs))
                        f *= math.prod(2.0 ** -emulator._scale_exp(r[1]) for r in recs)
                        if d.lsplit and d.rs[k]:
                            self.set_rec(d.rs[k], b, exp=exps[k], maxbits=0)
                prod = side[0] * side[1] * f
                if d.lsplit:
                    parts = prod.reshape(1 << d.nreg, 1 << d.lsplit, -1).sum(axis=(0, 2))
                    P = self.heap.view(d.partial, np.float64, d.nbatch << d.lsplit)
                    P[b << d.lsplit:(b + 1) << d.lsplit] = parts
                    self.gemm_partials.add(d.partial)
                    continue
                val = self.dt(prod.sum())
                self.heap.view(d.c + b * d.cb * esz, self.dt, 1)[0] = val
                if self.scaled:
                    self.set_rec(d.cs, b, exp=sum(exps), maxbits=int(np.abs(val).view(np.uint32)))

    def op_15(self, L):
        # block by block: the streams' tasks level by level; LDS starts as NaN, every tensor
        # is read only after its level, and every wave meets the same barriers
        esz, waves = self.dt().itemsize, int(L.iaux0)
        for i in range(L.count):
            d = self.heap.read_struct(_lib.TreeDesc, L.descs + i * ctypes.sizeof(_lib.TreeDesc))
            st = self.heap.view(d.tasks, np.uint32, waves * d.ntask).reshape(waves, -1).astype(np.int64)
            bar = st >> 31
            assert np.all(bar == bar[0]) and np.all(bar[:, -1] == 1)
            ops = self.heap.view(d.ops, np.uint32, _lib.TO_TREE_WORDS * (1 + int((st & 0xffff).max())))
            ops = ops.reshape(-1, _lib.TO_TREE_WORDS)
            ops = ops.astype(np.int64)
            for batch in range(d.nblocks):
                data = np.full((L.lds - (8 * d.nslots + 15) // 16 * 16) // esz, np.nan, dtype=self.dt)
                recs = [[0, 0.0] for _ in range(d.nslots)]
                pending, done = [], set()
                for col in range(d.ntask):
                    for t in st[:, col]:
                        if t & _lib.TO_TREE_IDLE:
                            continue
                        k, c, step = int(t & 0xffff), int(t >> 16 & 127), 1 << int(t >> 23 & 15)
                        for chunk in range(c, 1 << int(ops[k][0] >> 12 & 15), step):
                            assert (k, chunk) not in done
                            done.add((k, chunk))
                            self._tree_task(d, ops[k], chunk, batch, data, recs, pending)
                    if bar[0, col]:
                        for write in pending:
                            write()
                        pending = []
                assert not pending
                assert len(done) == sum(1 << int(o[0] >> 12 & 15) for o in ops)
                self.operands = getattr(self, "operands", set()) | {int(o[0] >> 16 & 3) + 1 for o in ops}

    def _tree_task(self, d, op, chunk, batch, data, recs, pending):
        head = int(op[0])
        lo, lk, nloop, nchunk = head & 15, head >> 4 & 15, head >> 8 & 15, head >> 12 & 15
        nops = (head >> 16 & 3) + 1
        assert lo + lk <= 6 and 6 + nchunk + nloop <= 16
        assert nops <= 2 or (nchunk == 0 and nloop <= 2)
        assert nops >= 2
        esz = self.dt().itemsize
        prod, e, f = 1.0, 0, 1.0
        for j in list(range(nops)) + [4]:
            bits = op[64 + 16 * j:80 + 16 * j] if j < 4 else op[32:48]
            assert not np.any(bits[lo + lk:6])
            assert np.array_equal(op[128 + 64 * j:192 + 64 * j], _spread(bits, 0, 6))
            o = _spread(bits, 0, lo) + sum(int(bits[6 + b]) for b in range(nchunk) if chunk >> b & 1)
            k = (_spread(bits, lo, lk)[:, None] + _spread(bits, 6 + nchunk, nloop)[None, :]).ravel()
            if j == 4:
                break
            idx = o[:, None] + k[None, :]
            addr = int(op[1 + 2 * j]) | int(op[2 + 2 * j]) << 32
            slot = int(op[16 + j])
            if head >> (20 + j) & 1:
                prod = prod * data[addr + idx].astype(np.float64)
                exp, bits_ = (recs[slot][0], int(np.float32(recs[slot][1]).view(np.uint32))) if self.scaled else (0, 0)
            else:
                src = self.heap.view(addr + batch * int(op[11 + j]) * esz, self.dt, int(idx.max()) + 1)
                prod = prod * src[idx].astype(np.float64)
                exp, bits_ = self.get_rec(d.recs, slot + (batch if head >> (25 + j) & 1 else 0)) if self.scaled else (0, 0)
            if self.scaled:
                e += exp + emulator._scale_exp(bits_)
                f *= 2.0 ** -emulator._scale_exp(bits_)
        assert not np.any(k)
        v = (prod.sum(axis=1) * f).astype(self.dt)
        assert np.all(np.isfinite(v))
        addr, slot = int(op[9]) | int(op[10]) << 32, int(op[20])

        def write():
            m = float(np.max(np.abs(v)))
            if head >> 24 & 1:
                data[addr + o] = v
                if self.scaled:
                    recs[slot][1] = max(recs[slot][1], m)
                    if chunk == 0:
                        recs[slot][0] = e
            else:
                self.heap.view(addr + batch * int(op[15]) * esz, self.dt, int(o.max()) + 1)[o] = v
                if self.scaled:
                    r = slot + (batch if head >> 29 & 1 else 0)
                    self.set_rec(d.recs, r, exp=e if chunk == 0 else None, maxbits=int(np.float32(m).view(np.uint32)))
        pending.append(write)

    def op_10(self, L):
        # products whose batch items share scale records in groups of 2^hlog
        for i in range(L.count):
            d = self.heap.read_struct(_lib.GemmDesc, L.descs + i * ctypes.sizeof(_lib.GemmDesc))
            if d.lsplit:
                assert d.hlog == 0 and L.count == 1
                super().op_10(L)
                continue
            M, N, K = 1 << d.mlog, 1 << d.nlog, 1 << d.klog
            esz = self.dt().itemsize
            cidx = np.arange(M)[:, None] * d.ldcm + np.arange(N)[None, :] * d.ldcn
            for b in range(d.nbatch):
                A = self.heap.view(d.a + b * d.ab * esz, self.dt, M * K).reshape(M, K).astype(np.float64)
                B = self.heap.view(d.b + b * d.bb * esz, self.dt, N * K).reshape(N, K).astype(np.float64)
                e, f, r = 0, 1.0, b >> d.hlog
                if self.scaled:
                    for rec in (self.get_rec(d.as_, r * d.asb), self.get_rec(d.bs, r * d.bsb)):
                        e += rec[0] + emulator._scale_exp(rec[1])
                        f *= 2.0 ** -emulator._scale_exp(rec[1])
                Cm = ((A @ B.T) * f).astype(self.dt)
                self.heap.view(d.c + b * d.cb * esz, self.dt, M * N)[cidx] = Cm
                if self.scaled:
                    m = np.float32(np.max(np.abs(Cm)))
                    self.set_rec(d.cs, r, exp=e, maxbits=int(m.view(np.uint32)))


class _Host:
    """What ``HipAPI._plan_inputs`` needs of an API, without a device."""

    def __init__(self, device_leaves=True):
        self._device_leaves = device_leaves

    def create_tensor(self, shape, default_value=None):
        return np.empty(shape) if default_value is None else np.full(shape, default_value, dtype=np.float64)

    reshape = staticmethod(np.reshape)

    @staticmethod
    def transpose(t, perm):
        return np.transpose(t, axes=perm)


def plan_inputs(plan, device_leaves=True):
    return hip_api.HipAPI._plan_inputs(_Host(device_leaves), plan, None)


def emulate(plan, et, W, device_leaves=True, group_levels=True, **kw):
    total, tree, tables, G = plan_inputs(plan, device_leaves)
    folded = fold.analyse(tree, tables, 8 if et == _lib.TO_F64 else 4, **kw)
    heap = emulator.Heap()
    prog = fold.compile_program(folded, tables, G, et, W, heap.alloc, group_levels, heap.alloc)
    for buf, data in ((prog.table, prog.table_host), (prog.coef, prog.coef_host), (prog.blob, prog.blob_host)):
        heap.write(buf, data.tobytes())
    if et == _lib.TO_F32S:
        heap.write(prog.recs, schedule.rec_init_bytes(prog))
    heap.write(prog.params, np.array([0, total, 0, 1], dtype=np.int64).tobytes())
    heap.write(prog.accum, bytes(_lib.Accum()))
    emu = FoldEmulator(heap, et)
    emu.run(prog.build)
    for run in range(2):  # a second run starts its sum anew
        emu.run(prog.prologue)
        if not prog.root_const:
            for _ in range(-(-total // W)):
                emu.run(prog.wave)
        acc = heap.read_struct(_lib.Accum, prog.host_accum.data_ptr())
        assert bytes(acc) == bytes(heap.read_struct(_lib.Accum, prog.accum.data_ptr())) and acc.count == total
    fm, fe = prog.leaf_factor
    return math.ldexp(acc.mant * fm, acc.exp + fe), prog, emu


@pytest.mark.parametrize("path", SMALL, ids=[os.path.basename(p)[:-5] for p in SMALL])
@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_fixture_folded(path, et, tol):
    doc = json.load(open(path))
    plan = plan_io.plan_from_dict(doc)
    want = numpy_oracle.contract_sliced(doc)
    total = 1 << len(plan.groups_to_slice)
    for W in sorted({1, 3, total}):
        got, prog, emu = emulate(plan, et, W)
        assert got == pytest.approx(want, rel=tol)
        assert emu.operands >= {2, 3, 4}
        assert prog.stats["tree_joins"] > prog.stats["joins"] // 2
    got, _, _ = emulate(plan, et, total, device_leaves=False, group_levels=False, regroup=False)
    assert got == pytest.approx(want, rel=tol)


@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_batch_folded(et, tol):
    # uneven instances in one grouped schedule: programs, and joins outside them (LDS for the
    # programs is kept so small that many are), grouped launches with block maps
    esize = 8 if et == _lib.TO_F64 else 4
    plans = [_formula_plan("vc", n, seed, 0) for seed, n in enumerate([10, 16, 24, 40, 30, 20, 18, 56])]
    plans.append(_formula_plan("vc", 70, 0, 0))  # (holds a product)
    wants = [numpy_oracle.contract_sliced(plan_io.plan_to_dict(p)) for p in plans]
    for lds, bits in ((64 * 1024, 16), (256, 5)):
        saved = fold.TREE_LDS_BATCH, fold.TREE_BITS
        fold.TREE_LDS_BATCH, fold.TREE_BITS = lds, bits
        try:
            per = fold.analyse_batch([plan_inputs(p)[1:3] for p in plans], esize)
        finally:
            fold.TREE_LDS_BATCH, fold.TREE_BITS = saved
        # what a program makes for a product is stored as the product reads it
        stored = [not n.geom["var"][key] for p in per for n in p["nodes"]
                  if not n.is_leaf and n.geom["var"]["kind"] == "gemm"
                  for key, i in (("perm_x", n.geom["X"]), ("perm_y", n.geom["Y"]))
                  if any(i in g.members for g in p["programs"])]
        assert all(stored) and (stored or bits == 5)
        heap = emulator.Heap()
        arena = heap.alloc(sum(p["region"] for p in per))
        prog = fold.compile_batch(per, et, heap.alloc, arena, heap.alloc)
        for buf, data in ((prog.table, prog.table_host), (prog.blob, prog.blob_host)):
            heap.write(buf, data.tobytes())
        if et == _lib.TO_F32S:
            from tensororder_amd import batch

            heap.write(prog.recs, batch.rec_init_bytes(prog))
        emu = FoldEmulator(heap, et)
        emu.run(prog.build)
        for _ in range(2):  # replays
            emu.run(prog.launches)
            for i, want in enumerate(wants):
                acc = heap.read_struct(_lib.Accum, prog.accum.data_ptr() + i * ctypes.sizeof(_lib.Accum))
                fm, fe = prog.leaf_factors[i]
                assert math.ldexp(acc.mant * fm, acc.exp + fe) == pytest.approx(want, rel=tol)
        assert emu.maps_checked > 0
        assert (prog.stats["steps"] > 4) == (bits == 5)


def _formula_plan(kind, n, seed, slices):
    text = vertex_cover_cnf(n, seed, True) if kind == "vc" else random_3cnf(n, int(1.9 * n), seed, True)
    net = network.cnf_count(parse_dimacs_text(text, "cachet"))
    plan = planners.best_plan(net, "line" if kind == "vc" else "factor", solver=None, seed=seed)
    ALL_SLICERS["greedy_mem"].slice_until(plan, slices=slices)
    return plan


@pytest.mark.parametrize("kind,n,slices", [("vc", 14, 0), ("vc", 26, 2), ("cnf", 12, 0), ("cnf", 18, 3), ("cnf", 25, 1)])
@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_random_formulas_folded(kind, n, slices, et, tol):
    for seed in range(3):
        plan = _formula_plan(kind, n, seed, slices)
        want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
        got, prog, _ = emulate(plan, et, 1 << slices)
        assert got == pytest.approx(want, rel=tol)


def test_unused_variables_and_repeated_leaves_folded():
    from test_emulator import unused_variable_plans

    for name, plan in unused_variable_plans():
        want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
        for et, tol in ((_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)):
            assert emulate(plan, et, 1)[0] == pytest.approx(want, rel=tol), name


def test_early_contracted_plan_folded():
    from test_emulator import early_contracted_plan

    plan, want = early_contracted_plan(4)
    for et, tol in ((_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)):
        assert emulate(plan, et, 8)[0] == pytest.approx(want, rel=tol)


def test_folded_tensors_hold_each_variable_once():
    # rank by rank: a folded tensor never holds more variables than the walk's tensor has
    # axes, and the large formula's plan shrinks as its COPY structure says
    doc = json.load(open(os.path.join(HERE, "golden", "cnf70_factor_s12.json")))
    plan = plan_io.plan_from_dict(doc)
    _, tree, tables, _ = plan_inputs(plan)
    nodes, missing = fold.analyse(tree, tables, 4)
    assert missing == 0
    assert max(n.rank for n in nodes) <= 22 < doc["meta"]["maxrank"]
    assert sum(fold.join_traffic(n, nodes, 1, 4)[1] for n in nodes if not n.is_leaf) < 2 ** 28


# (X-only, Y-only, kept shared, summed shared, X-only summed, slices, X sliced, Y sliced,
#  shuffled): the general form below and above 256 outputs, with shared thread bits and with
#  blocks sharing a sum; the 16-byte form with 0..3 (and more) register bits, Y holding none,
#  both or one of the lowest two variables; the streamed operand the smaller one ("yy", "yh",
#  "hy": the outputs' lowest variables by kind); odd slice counts
JOINS = [(0, 0, 0, 0, 0, 1, 1, 1, 0), (2, 1, 1, 1, 0, 3, 1, 1, 1), (3, 2, 2, 2, 1, 5, 1, 0, 1), (0, 0, 3, 9, 0, 2, 1, 1, 0),
         (0, 0, 0, 16, 0, 1, 1, 1, 0), (1, 0, 1, 14, 0, 3, 1, 1, 1), (4, 5, 1, 6, 0, 1, 1, 1, 1), (10, 0, 0, 0, 0, 1, 1, 1, 0),
         (11, 0, 2, 1, 0, 2, 1, 0, 0), (9, 1, 4, 2, 0, 3, 1, 1, 0), (10, 2, 2, 3, 0, 1, 1, 1, 0), (8, 3, 3, 1, 0, 7, 1, 0, 0),
         (4, 6, 5, 2, 0, 65, 1, 1, 1), (4, 2, 9, 1, 0, 33, 1, 0, 1), (1, 1, 13, 1, 1, 9, 1, 1, 1),
         (2, 0, 13, 0, 0, 9, 1, 1, 1), (0, 0, 0, 18, 0, 3, 1, 1, 0), (1, 0, 2, 11, 0, 2, 1, 0, 0),
         (9, 5, 3, 2, 0, 2, 1, 1, 0), (0, 0, 13, 1, 0, 3, 1, 1, 0), (1, 0, 12, 2, 0, 2, 1, 1, 0), (12, 1, 1, 4, 0, 3, 1, 1, 0),
         (6, 5, 4, 3, 0, 5, 1, 1, "yy"), (5, 4, 6, 0, 1, 3, 1, 0, "yh"), (6, 5, 4, 3, 0, 5, 1, 1, "yyxx"), (2, 8, 3, 1, 0, 3, 0, 1, "yyxx"), (3, 2, 8, 1, 0, 65, 1, 1, "hy"),
         (4, 3, 6, 2, 0, 3, 0, 1, "hx"), (9, 0, 3, 1, 1, 2, 1, 1, "xh"), (2, 2, 9, 2, 0, 9, 1, 1, "hh"), (4, 3, 7, 2, 0, 3, 1, 0, "hhr")]


def _join(case, et, alloc, write, rng):
    """One folded join compiled by ``fold.choose``: (records, node list, data, result)."""
    xo, yo, kept, s, xs, W, xw, yw, shuffled = case
    esize = 8 if et == _lib.TO_F64 else 4
    dt = np.float64 if esize == 8 else np.float32
    names = ["x%d" % i for i in range(xo)] + ["h%d" % i for i in range(kept)]
    if kept and not shuffled and rng.integers(2):  # kept variables lowest: Y's lowest too
        names = names[xo:] + names[:xo]
    ks = ["k%d" % i for i in range(s)] + ["q%d" % i for i in range(xs)]
    xv = names + ks if s < fold.DOT_MIN_SHARED else ks + names  # long sums: shared lowest
    yv = [v for v in xv if v[0] in "hk"] + ["y%d" % i for i in range(yo)]
    out = names + ["y%d" % i for i in range(yo)]
    if shuffled:
        for v in (xv, yv, out):
            rng.shuffle(v)
    if isinstance(shuffled, str):  # the lowest two variables by kind, as in the plan's one order
        low = [u + str(shuffled[:i].count(u)) for i, u in enumerate(shuffled.rstrip("r"))]
        one = low + [v for v in out if v not in low] + sorted(set(xv + yv) - set(out))
        xv, yv, out = ([v for v in one if v in vs] for vs in (xv, yv, out))
        if shuffled.endswith("r"):  # (a leaf's axes lie as they are)
            yv.reverse()
    nodes = []
    for i, (vs, batched) in enumerate(((xv, xw), (yv, yw), (out, xw or yw))):
        n = fold.FNode(i)
        n.is_leaf, n.batched, n.order = i < 2, bool(batched), list(vs)
        n.order0, n.rank, n.left, n.right = n.order, len(vs), 0, 1
        n.off = {v: 1 << j for j, v in enumerate(vs)}
        nodes.append(n)
    X, Y, C = nodes
    C.ksum = set(xv + yv) - set(out)
    fold.choose(C, nodes, W, esize)
    data, recs = {}, {}
    for n in (X, Y, C):
        items = W if n.batched else 1
        n.bstride = (1 << n.rank) if n.batched else 0
        n.rec_stride = 1 if n.batched else 0
        n.ptr = alloc(items * esize << n.rank)
        recs[n.idx] = alloc(16 * items)
        if n is not C:
            data[n.idx] = rng.uniform(0.25, 1.0, (items, 1 << n.rank)).astype(dt)
            write(n.ptr, data[n.idx].tobytes())
            write(recs[n.idx], b"".join(
                bytes(_lib.ScaleRec(exp=3 - b, maxbits=int(np.abs(data[n.idx][b]).max().astype(np.float32).view(np.uint32))))
                for b in range(items)))
        else:
            write(recs[n.idx], bytes(16 * items))
    v = C.geom["var"]
    scratch = {"partial": (alloc(v["nout"] * v["nsplit"] * 8), 0)} if v.get("lsplit") else {}
    records = fold.join_records(C, nodes, W, esize, esize == 4, 0, scratch, lambda n: recs[n.idx], (0, 0))
    # float64 result, indexed by C's own bits
    def off(n, vs):
        o = np.zeros(1, dtype=np.int64)
        for u in vs:
            o = np.concatenate([o, o + n.off.get(u, 0)])
        return o
    ks = sorted(C.ksum)
    ox, oy = (off(n, C.order)[:, None] + off(n, ks)[None, :] for n in (X, Y))
    want = []
    for b in range(W if C.batched else 1):
        x, y = (data[n.idx][b if n.batched else 0].astype(np.float64) for n in (X, Y))
        want.append((x[ox] * y[oy]).sum(axis=1) * 2.0 ** (sum(3 - (b if n.batched else 0) for n in (X, Y)) if esize == 4 else 0))
    return records, nodes, recs, np.array(want)


def _launches(records, alloc, write):
    out = []
    for kind, op, variant, lds, st, nblk in records:
        st.block0 = 0
        at = alloc(len(bytes(st)))
        write(at, bytes(st))
        out.append(_lib.Launch(op=op, variant=variant, count=1, grid=nblk, lds=lds, descs=at))
    return out


def _check(case, et, got, rec, want, rtol=1e-13):
    # products of floats are exact in the double sums: one rounding, at the store
    dt = np.float64 if et == _lib.TO_F64 else np.float32
    for b in range(want.shape[0]):
        scale = 2.0 ** int(rec[b].exp) if et == _lib.TO_F32S else 1.0
        np.testing.assert_allclose(got[b].astype(np.float64) * scale, want[b], rtol=rtol if dt == np.float64 else 1.2e-7)
        if et == _lib.TO_F32S:
            assert rec[b].maxbits == int(np.abs(got[b]).max().view(np.uint32))


@pytest.mark.parametrize("et", [_lib.TO_F64, _lib.TO_F32S], ids=["f64", "f32s"])
def test_every_form_emulated(et):
    forms = set()
    for i, case in enumerate(JOINS):
        heap = emulator.Heap(1 << 27)
        ptr = {}

        def alloc(n):
            b = heap.alloc(n)
            ptr[b.data_ptr()] = b
            return b.data_ptr()

        def write(at, data):
            heap.write(ptr[at], data)

        records, nodes, recs, want = _join(case, et, alloc, write, np.random.default_rng(i))
        emu = FoldEmulator(heap, et)
        emu.run(_launches(records, alloc, write))
        forms |= emu.forms
        if any(r[0] == "finish" for r in records):
            forms.add("split")
        C = nodes[2]
        items = want.shape[0]
        got = heap.view(C.ptr, emu.dt, items << C.rank).reshape(items, -1)
        _check(case, et, got, [heap.read_struct(_lib.ScaleRec, recs[2] + 16 * b) for b in range(items)], want)
    assert {f & 15 for f in forms if f != "split" and f & _lib.TO_FOLD_VEC} == {0, 1, 2, 3}
    assert {f >> 4 & 15 for f in forms if f != "split" and f & _lib.TO_FOLD_VEC} == {0, 1, 2, 3, 4, 5}
    assert "split" in forms and _lib.TO_FOLD_ANY in forms and _lib.TO_FOLD_DOT in forms
    assert {f for f in forms if f != "split" and f & _lib.TO_FOLD_REG} == {
        _lib.TO_FOLD_REG | a << 4 | b for a, b in fold.REG_TILES}


@pytest.mark.gpu
@pytest.mark.parametrize("et", [_lib.TO_F64, _lib.TO_F32S], ids=["f64", "f32s"])
def test_every_form_on_the_device(et):
    import torch

    api = hip_api.HipAPI() if et == _lib.TO_F64 else hip_api.HipF32API()
    for i, case in enumerate(JOINS):
        _say("case folded join", et, case)
        ptr = {}

        def alloc(n):
            t = torch.full((n,), 255, dtype=torch.uint8, device="cuda")  # NaN where nothing is written
            ptr[t.data_ptr()] = t
            return t.data_ptr()

        def write(at, data):
            ptr[at][:len(data)] = torch.frombuffer(bytearray(data), dtype=torch.uint8).cuda()

        records, nodes, recs, want = _join(case, et, alloc, write, np.random.default_rng(i))
        launches = _launches(records, alloc, write)
        torch.cuda.synchronize()
        api._run(launches)
        api.synchronize()
        items, C = want.shape[0], nodes[2]
        dt = np.float64 if et == _lib.TO_F64 else np.float32
        got = ptr[C.ptr].cpu().numpy().view(dt).reshape(items, -1)
        raw = ptr[recs[2]].cpu().numpy().tobytes()
        _check(case, et, got, [_lib.ScaleRec.from_buffer_copy(raw[16 * b:16 * b + 16]) for b in range(items)], want)


@pytest.mark.gpu
@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)], ids=["f64", "f32s"])
def test_folded_and_edge_walk_agree_on_the_device(et, tol):
    # the folded executor against the walk over edges (tables without their COPY mark), on
    # plans with products whose kept variables are batch items
    api = hip_api.HipAPI() if et == _lib.TO_F64 else hip_api.HipF32API()
    for kind, n, seed, slices in (("vc", 70, 2, 0), ("cnf", 34, 4, 2), ("cnf", 40, 1, 3)):
        _say("case folded vs walk", kind, n, slices, et)
        plan = _formula_plan(kind, n, seed, slices)
        total, tree, tables, G = api._plan_inputs(plan, None)
        exe = api._compile(tree, tables, G, total)
        got = [exe.run().value for _ in range(3)]
        exe.close()
        for t in tables.values():
            t.copy = None
        exe = api._compile(tree, tables, G, total)
        want = exe.run().value
        exe.close()
        assert got == pytest.approx([want] * 3, rel=tol)


@pytest.mark.gpu
def test_options_on_folded_plans(tmp_path, monkeypatch):
    # the autotune option times the products of a folded plan; the cost model's records are
    # those of the joins edge by edge
    from tensororder_amd import autotune, train_costmodel

    monkeypatch.setenv("TENSORORDER_TUNE_CACHE", str(tmp_path / "tune.json"))
    f = parse_dimacs_text(vertex_cover_cnf(80, 3, True), "cachet")
    plan = planners.candidate_plans(network.cnf_count(f), "line", [11])[0]
    api = hip_api.HipF32API()
    want = api.contract_sliced(plan)
    saved = dict(schedule.TUNED)
    try:
        schedule.TUNED.clear()
        api.add_argument("autotune", True)
        got = api.contract_sliced(plan)
        total, tree, tables, groups = api._plan_inputs(plan, None)
        nodes, _ = fold.analyse(tree, tables, 4)
        fold.choose_all(nodes, 1, 4)
        products = {autotune.gemm_key(4, n.geom["fx"], n.geom["fy"], n.geom["s"], 1 << n.geom["var"]["hlog"])
                    for n in nodes if not n.is_leaf and n.geom["var"]["kind"] == "gemm"}
        assert products and products <= set(schedule.TUNED)
    finally:
        schedule.TUNED.clear()
        schedule.TUNED.update(saved)
    assert got == pytest.approx(want, rel=1e-5)
    x, y = train_costmodel.timed_records(api, plan)
    assert x.shape[0] == y.shape[0] > 0 and x.shape[1] == 16 and np.isfinite(x).all() and np.isfinite(y).all()


def test_wide_joins_run_edge_by_edge(monkeypatch):
    # a join over more variables than a descriptor holds, or a plan whose folded arena would
    # not fit: the batch size says so (0), the unfolded path takes the plan
    f = parse_dimacs_text(random_3cnf(24, 46, 5, True), "cachet")
    plan = planners.candidate_plans(network.cnf_count(f), "factor", [11])[0]
    total, tree, tables = plan_inputs(plan)[:3]
    folded = fold.analyse(tree, tables, 8)

    class Api:
        _esize, _regroup, _max_batch, budget = 8, True, 64, 1 << 30
        choose_batch = None

        def _budget(self):
            return self.budget

    api = Api()
    assert hip_api.HipAPI.choose_folded_batch(api, folded, tree, tables, 1) == 1
    with monkeypatch.context() as m:
        m.setattr(fold._lib, "FOLD_BITS", 6)
        assert hip_api.HipAPI.choose_folded_batch(api, folded, tree, tables, 1) == 0
        assert fold.analyse_batch([(tree, tables)], 8) is None
    monkeypatch.setattr(fold, "peak_bytes", lambda *a: 2 << 30)
    assert hip_api.HipAPI.choose_folded_batch(api, folded, tree, tables, 1) == 0


@pytest.mark.gpu
def test_ends_of_runs_on_the_device():
    # a run's end is seen by a word its sum writes, that of other calls by a signal: runs
    # queued together, launches run outside the executable between runs, and several threads
    # waiting on one API
    import threading

    plan = plan_io.plan_from_dict(json.load(open(os.path.join(HERE, "golden", "cnf20_factor_s4.json"))))
    want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
    for graph in (True, False):
        api = hip_api.HipAPI()
        api.add_argument("graph", graph)
        api.add_argument("max_batch", 4)
        exe = api.prepare(plan)
        for queued in (1, 3, 2):
            for _ in range(queued):
                exe.enqueue()
            r = exe.result()
            assert r.value == pytest.approx(want, rel=1e-12) and r.slices == exe.total
            api._run(exe.step_launches + exe.wave_launches * exe.nwaves)
            api.synchronize()
            assert exe.result().mant == r.mant
        exe.close()
    rng = np.random.default_rng(0)
    pairs = [(rng.random((2,) * 12), rng.random((2,) * 10)) for _ in range(4)]
    got = [None] * 4

    def work(i):
        for _ in range(20):
            got[i] = api.tensordot(*pairs[i], ([0, 1, 2], [2, 1, 0]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for (a, b), out in zip(pairs, got):
        out = out.numpy() if hasattr(out, "numpy") else out
        np.testing.assert_allclose(out, np.tensordot(a, b, ([0, 1, 2], [2, 1, 0])), rtol=1e-12)


# dot products with their operands' joins inside (each with the lowest variables in no small
# operand, and as listed): variables both large operands have, that only
# the first / only the second has, summed by the joins; slices; whether each operand has them;
# the lowest two variables in the small operands: none, both lowest, both, first, second
PAIRS = [(14, 0, 0, 0, 0, 1, "xyzw", "nn"), (15, 0, 1, 1, 0, 3, "xyzw", "vs"), (13, 2, 1, 2, 1, 5, "xyz", "sv"),
         (12, 1, 3, 1, 1, 2, "xzw", "ss"), (13, 1, 0, 2, 0, 33, "xyzw", "nf"), (13, 3, 1, 2, 2, 2, "xyzw", "bv"),
         (10, 4, 1, 2, 1, 4097, "xyzw", "sn"), (16, 0, 0, 1, None, 2, "xyz", "s"), (14, 0, 1, 2, None, 3, "xyz", "v")]


PAIRS += [case[:7] + ("n" * len(case[7]),) for case in PAIRS] + [(13, 1, 1, 1, 1, 3, "xyzw", "nn"), (14, 1, 0, 2, 2, 1, "xw", "nn"),
                                                              (14, 0, 0, 0, 0, 2, "yz", "sn")]


def _pair(case, et, alloc, write, rng):
    """A root dot product with its joins compiled by ``fold.choose_all``, as ``_join``."""
    body, r0, r1, na, nb, W, sliced, lows = case
    esize = 8 if et == _lib.TO_F64 else 4
    dt = np.float64 if esize == 8 else np.float32
    big = ["v%d" % i for i in range(body)]
    ya_only, yb_only = ["s%d" % i for i in range(r0)], ["t%d" % i for i in range(r1)]
    sums = [["i%d" % i for i in range(na)], ["j%d" % i for i in range(nb or 0)]]
    out = big + ya_only + yb_only

    def small(how, own):
        mid = [str(v) for v in rng.permutation(big[2:])[:3]]
        low = {"n": [], "v": big[:2], "s": [], "f": [], "b": []}[how]
        rest = mid + own + {"s": big[1:2], "f": big[:1], "b": big[:2]}.get(how, [])
        rng.shuffle(rest)
        return low + rest

    def large(own):
        rest = big[2:] + own
        rng.shuffle(rest)
        return big[:2] + rest

    specs = [(large(yb_only + sums[0]), "x" in sliced), (small(lows[0], ya_only + sums[0]), "y" in sliced)]
    if nb is not None:
        specs += [(large(ya_only + sums[1]), "z" in sliced), (small(lows[1], yb_only + sums[1]), "w" in sliced)]
    else:  # the other operand is stored
        specs += [(big + yb_only, "z" in sliced)]
    nodes = []

    def add(order, batched, left=-1, right=-1, ksum=()):
        n = fold.FNode(len(nodes))
        n.is_leaf, n.batched, n.order, n.order0 = left < 0, bool(batched), list(order), list(order)
        n.rank, n.left, n.right, n.ksum = len(order), left, right, set(ksum)
        n.off = {v: 1 << j for j, v in enumerate(order)}
        nodes.append(n)
        return n.idx

    leaves = [add(*sp) for sp in specs]
    a = add(out, True, leaves[0], leaves[1], sums[0])
    b = add(out, True, leaves[2], leaves[3], sums[1]) if nb is not None else leaves[2]
    add([], True, a, b, out)
    fold.choose_all(nodes, W, esize)
    data, recs = {}, {}
    for n in nodes:
        items = W if n.batched else 1
        n.bstride = (1 << n.rank) if n.batched else 0
        n.rec_stride = 1 if n.batched else 0
        recs[n.idx] = alloc(16 * items)
        write(recs[n.idx], bytes(16 * items))
        if n.is_leaf or n is nodes[-1]:
            n.ptr = alloc(items * esize << n.rank)
        if n.is_leaf:
            data[n.idx] = rng.uniform(0.25, 1.0, (items, 1 << n.rank)).astype(dt)
            write(n.ptr, data[n.idx].tobytes())
            write(recs[n.idx], b"".join(bytes(_lib.ScaleRec(exp=3 - k % 7, maxbits=int(
                np.abs(data[n.idx][k]).max().astype(np.float32).view(np.uint32)))) for k in range(items)))
    root = nodes[-1]
    v = root.geom["var"]
    assert v["kind"] == "pair" and nodes[a].geom["var"]["kind"] == "fused"
    one = alloc(256)
    write(one, dt(1).tobytes())
    scratch = {"partial": (alloc(v["nout"] * v["nsplit"] * 8), 0)} if v.get("lsplit") else {}
    records = fold.join_records(root, nodes, W, esize, esize == 4, 0, scratch, lambda n: recs[n.idx], (one, 0))
    want = []
    for k in range(min(W, 5)):
        terms = [(data[i][k if nodes[i].batched else 0].astype(np.float64).reshape((2,) * nodes[i].rank),
                  nodes[i].order[::-1]) for i in leaves]
        number = {u: j for j, u in enumerate(sorted({u for _, vs in terms for u in vs}))}
        halves = []
        for part in (terms[:2], terms[2:]):
            args = [x for t, vs in part for x in (t, [number[u] for u in vs])]
            halves.append(np.einsum(*args, [number[u] for u in out]))
        e = sum(3 - (k % 7 if nodes[i].batched else 0) for i in leaves) if esize == 4 else 0
        want.append([(halves[0] * halves[1]).sum() * 2.0 ** e])
    return records, nodes, recs, np.array(want)


@pytest.mark.parametrize("et", [_lib.TO_F64, _lib.TO_F32S], ids=["f64", "f32s"])
def test_fused_dot_products_emulated(et):
    forms = set()
    for i, case in enumerate(PAIRS):
        if case[5] > 100:
            continue  # whole blocks of slices: on the device
        heap = emulator.Heap(1 << 26)
        ptr = {}

        def alloc(n):
            b = heap.alloc(n)
            ptr[b.data_ptr()] = b
            return b.data_ptr()

        def write(at, data):
            heap.write(ptr[at], data)

        records, nodes, recs, want = _pair(case, et, alloc, write, np.random.default_rng(i))
        emu = FoldEmulator(heap, et)
        emu.run(_launches(records, alloc, write))
        forms |= emu.forms
        got = heap.view(nodes[-1].ptr, emu.dt, case[5]).reshape(-1, 1)[:len(want)]
        rec = [heap.read_struct(_lib.ScaleRec, recs[nodes[-1].idx] + 16 * b) for b in range(len(want))]
        _check(case, et, got, rec, want, 1e-12)
    assert {f[1] for f in forms if isinstance(f, tuple)} == {
        k | one for k in (0x00, 0x10, 0x11, 0x20, 0x21, 0x22) for one in (0, _lib.TO_PAIR_ONE)}


@pytest.mark.gpu
@pytest.mark.parametrize("et", [_lib.TO_F64, _lib.TO_F32S], ids=["f64", "f32s"])
def test_fused_dot_products_on_the_device(et):
    import torch

    api = hip_api.HipAPI() if et == _lib.TO_F64 else hip_api.HipF32API()
    for i, case in enumerate(PAIRS):
        _say("case fused dot", et, case)
        ptr = {}

        def alloc(n):
            t = torch.full((n,), 255, dtype=torch.uint8, device="cuda")
            ptr[t.data_ptr()] = t
            return t.data_ptr()

        def write(at, data):
            ptr[at][:len(data)] = torch.frombuffer(bytearray(data), dtype=torch.uint8).cuda()

        records, nodes, recs, want = _pair(case, et, alloc, write, np.random.default_rng(i))
        launches = _launches(records, alloc, write)
        torch.cuda.synchronize()
        api._run(launches)
        api.synchronize()
        dt = np.float64 if et == _lib.TO_F64 else np.float32
        got = ptr[nodes[-1].ptr].cpu().numpy().view(dt).reshape(-1, 1)[:len(want)]
        raw = ptr[recs[nodes[-1].idx]].cpu().numpy().tobytes()
        rec = [_lib.ScaleRec.from_buffer_copy(raw[16 * b:16 * b + 16]) for b in range(len(want))]
        _check(case, et, got, rec, want, 1e-12)


def _halves_plan(seed, slices):
    """A plan whose root is the dot product of two halves, each a large tensor absorbing a
    small one: dense tensors tied by COPY tensors of 12 to 14 variables."""
    from tensororder_amd.network import BuiltTensor, TensorNetwork, VariableTensor
    from tensororder_amd.plan import SlicedExecutionPlan
    from tensororder_amd.tree import TreeContext

    rng = np.random.default_rng(seed)
    big = ["v%d" % i for i in range(13)]
    tensors = [big + ["i"], ["i", "s"] + big[3:6], big[:11] + ["s", "j"], ["j"] + big[9:13]]
    net, ends = TensorNetwork(), {}
    for vs in tensors:
        # the first variables are the lowest bits of the large tensors, as the executor orders its own
        vs = [str(v) for v in rng.permutation(vs[2:])] + vs[1::-1] if len(vs) > 6 else vs
        for v, end in zip(vs, net.add_node(BuiltTensor(rng.uniform(0.5, 1.0, (2,) * len(vs))))):
            ends.setdefault(v, []).append(end)
    copies = {}
    for v, held in ends.items():
        at = net.add_node(VariableTensor(len(held), 1, 1 if v != "v5" else 0.5))
        copies[v] = at[0][0]
        for (t, ax), end in zip(held, at):
            net.connect(t, ax, *end)
    ctx = TreeContext()
    halves = []
    for a, b, inner in ((0, 1, "i"), (2, 3, "j")):
        # (the variable summed inside a half is tied before the small tensor comes)
        half = ctx.join(ctx.join(ctx.leaf(net, a), ctx.leaf(net, copies[inner])), ctx.leaf(net, b))
        halves.append(half)
    for v in copies:
        if v not in "ij":
            halves[0] = ctx.join(halves[0], ctx.leaf(net, copies[v]))
    plan = SlicedExecutionPlan(ctx.get_tree(ctx.join(*halves)), net)
    ALL_SLICERS["greedy_mem"].slice_until(plan, slices=slices)
    return plan


@pytest.mark.parametrize("et,tol", [(_lib.TO_F64, 1e-12), (_lib.TO_F32S, 1e-6)])
def test_fused_dot_products_in_plans(et, tol, monkeypatch):
    # whole plans, the rank from which joins are fused lowered
    monkeypatch.setattr(fold, "TREE_RANK", 9)
    fused = set()
    for seed in range(3):
        for slices in (0, 1, 2):
            plan = _halves_plan(seed, slices)
            want = numpy_oracle.contract_sliced(plan_io.plan_to_dict(plan))
            for W in {1, 1 << slices}:
                got, prog, emu = emulate(plan, et, W, device_leaves=False)
                assert got == pytest.approx(want, rel=tol)
                fused |= {(slices, f[1]) for f in emu.forms if isinstance(f, tuple)}
    assert {f[0] for f in fused} >= {0, 1} and {f[1] & 0xff for f in fused} == {0x11}


@pytest.mark.parametrize("cls", [hip_api.Executable, hip_api.BatchExecutable])
def test_dropped_runs_are_waited_for(cls):
    # the device writes an executable's host memory until its runs end: one that goes away, or
    # is closed, with a run nobody waited for waits first
    class Api:
        waits = 0

        def synchronize(self):
            Api.waits += 1

    for close in (False, True):
        exe = object.__new__(cls)
        exe.api, exe._graphs, exe._runs, exe._queued = Api(), [], [], 1
        before = Api.waits
        if close:
            exe.close()
            assert Api.waits == before + 1
        del exe
        assert Api.waits == before + 1
