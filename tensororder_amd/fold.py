"""Folded plans: a contraction tree whose COPY tensors are index identities.

A CNF network holds one COPY (variable) tensor per variable, split into pieces by the
planners, and every COPY tensor forces its edges equal
(``tensor_network_constructions.py:122-159``; the reference's own equivalence sets are
``find_equivalent_edges``, ``tensor_network.pyx:470-489``).  A tensordot walk stores one axis
per *edge*, so an intermediate that holds several edges of one variable is zero wherever they
differ.  Here such edges are one *variable* of the schedule:

* a tensor is indexed by the distinct variables of its free edges; a join may share a variable
  with its result (kept), sum it, or take it from one operand (``to_fold_desc``);
* a variable is summed at the lowest join that covers every leaf holding it;
* an unweighted COPY piece is a vector of ones and is dropped; a weight vector multiplies one
  leaf that holds its variable, wherever the tree had placed it;
* chains in which a large tensor absorbs small ones are reassociated by the bytes and products
  they cost, as in ``schedule.regroup_absorptions``.

Every tensor's bits are ordered by how late their variable is summed, the latest lowest.  The
order is one order for the whole plan, so the operands and the result of a join agree on it:
kept variables run along the lanes in all three, and the summed ones are the highest bits.
Dense joins (free ranges of >= 2^6 on both sides) go to the MFMA products, with the kept
shared variables as batch items.

The value is the same contraction; only structural zeros are left out.
"""

import ctypes
import math
import struct

import numpy as np

from . import _lib, schedule
from ._lib import LeafDesc, Launch

ALIGN = schedule.ALIGN

# Cost of a join for the reassociation (seconds): bytes at the rate of a large copy, products
# at the rate the folded kernels multiply and add (measured on the 4096-slice workload).
BYTES_PER_S = 5e12
PRODUCTS_PER_S = 8e12
GEMM_PRODUCTS_PER_S = 5e13
# operands of at most this many variables may be combined before a large tensor absorbs them
SMALL_RANK = 12
BIG_RANK = 10
# share of the cost of a join that runs once per slice, against one that runs once
BATCH_WEIGHT = 64.0
# threads a general-form launch should have before its shared range is left to one thread
ANY_MIN_THREADS_LOG = 17
MAX_ANY_BLOCKS = 8192
MAX_VEC_BLOCKS = 4096
MAX_REG_BITS = 3
# blocks of a fused dot product (four waves each; a CU holds eight blocks)
PAIR_MIN_BLOCKS_LOG = 13
# register tiles (variables only X has, only Y has), the first that a join has; it must leave
# this many outputs to threads
REG_TILES = ((2, 3), (2, 2), (1, 1), (2, 0))
REG_MIN_LOG = 16
# shared range from which a sum over few outputs takes four consecutive products per load
DOT_MIN_SHARED = 10
# programs run by one block per slice: joins over at most 2^TREE_BITS index values with
# results of at most 2^TREE_RANK entries, the intermediates in TREE_LDS bytes of LDS -- or
# TREE_LDS_MANY with TREE_WAVES_MANY waves, so that blocks share a CU, when there are enough
# slices to fill the chip
TREE_BITS = 16
TREE_RANK = 13
TREE_FAR_RANK = 9
TREE_FAR_BITS = 13
TREE_WAVES = 16
TREE_WAVES_MANY = 8
TREE_LDS = 120 * 1024
TREE_LDS_MANY = 40 * 1024
TREE_MANY = 512
# joins from which a program is fitted bit by bit as it grows
TREE_LONG = 256
# products of a program (a task word has 16 bits for its product)
TREE_PRODUCTS = 1 << 16
# a program of one join only up to this many index values (a launch of many blocks above)
TREE_LONE_BITS = 12
# joins of a program merged into one product: at most 4 operands, 64 outputs and 2^MERGE_LOOP
# products per output (each merge saves a level)
MERGE_LOOP = 2
# small operands of a product are stored by the join that makes them as the product reads them,
# whatever that does to its own stores: the launch that permuted them before the product took
# 17-19 us on a few tensors of 2^12 entries
WANT_ENTRIES = 1 << 20
# level launches are kept whatever they cost in memory up to this arena size
LEVEL_FREE_BYTES = 256 << 20

# bit b of lane l
_LANE_BITS = ((np.arange(64)[None, :] >> np.arange(6)[:, None]) & 1).astype(np.uint32)
# words of a product that hold the entries of its lane bits: operands 0-3, the result
_LANE_ENTRIES = np.array([at + b for at in (64, 80, 96, 112, 32) for b in range(6)])
_HEAD = struct.Struct("<QQQqqqQQQqqQ10i")
_BITS = struct.Struct("<%dI" % (3 * _lib.FOLD_BITS))


class FoldDesc:
    """A to_fold_desc under construction (``block0`` is set when a launch groups it)."""

    __slots__ = ("ptrs", "strides", "recs", "rec_strides", "partial", "nbatch", "block0", "nblocks", "roles", "bits")

    def __bytes__(self):
        lo, lk, ntile, nloop, lsplit, nreg = self.roles
        return _HEAD.pack(*self.ptrs, *self.strides, *self.recs, *self.rec_strides, self.partial, self.nbatch,
                          self.block0, self.nblocks, lo, lk, ntile, nloop, lsplit, nreg, 0) + _BITS.pack(*self.bits)


class TooWide(ValueError):
    """A join over more variables, or of a larger tensor, than a descriptor holds (offsets are
    32 bits), or more exponents than a program adds up: the plan runs edge by edge."""


OFFSET_BITS = 32
# nodes of an FP32-scaled plan: a program keeps its tensors' exponents in 32 bits, and a node adds
# less than 2^11 to them (a leaf's table lies between 2^-1074 and 2^1024)
EXPONENT_NODES = 1 << 20


class FNode:
    """A node of a folded plan.  ``order`` lists its variables from the lowest bit up and
    ``off`` maps each to the element offset it adds (several bits at once for a leaf that
    holds it on several axes); 2^rank entries are stored."""

    __slots__ = ("idx", "is_leaf", "tensor", "rank", "order", "order0", "want", "off", "batched", "left", "right", "parent",
                 "ksum", "geom", "buf", "ptr", "bstride", "rec", "rec_stride", "layout")

    def __init__(self, idx):
        self.idx = idx
        self.parent = -1
        self.want = None  # the order that the product reading it takes, where it is stored so
        self.buf = None
        self.rec = None
        self.rec_stride = 0
        self.layout = None  # at the root: the plan's layout, while the joins' forms are its own


class _T:
    """A subtree while the tree is built: ``open`` maps its unsummed variables to the number
    of leaves below that hold them, ``union`` counts the variables its join touches."""

    __slots__ = ("leaf", "open", "left", "right", "batched", "union", "cost")

    def __init__(self, leaf, open_, left=None, right=None, batched=False, union=0, cost=0.0):
        self.leaf, self.open, self.left, self.right = leaf, open_, left, right
        self.batched, self.union, self.cost = batched, union, cost


def has_copies(tables):
    """Whether a plan can be folded: its leaves include COPY tensors, each sliced on all of its
    edges by one group, or on none.  A COPY tensor sliced on a part of them ties what is left
    to the slice's value (and one sliced by two groups is 0 where these differ), which is no
    vector of ones and no identity of indices."""
    copies = [t for t in tables.values() if t.copy is not None]
    return bool(copies) and not any(t.rank if sum(map(bool, t.coef)) == 1 else t.batched for t in copies)


# 2.0^n of n variables (a plan of far more is refused for its memory)
_POWERS = [2.0 ** n for n in range(900)]


def _power(n):
    return _POWERS[n if n < 900 else -1]


def _join_cost(left, right, union, out, batched, esize):
    lx, ly = len(left.open), len(right.open)
    c = esize * (_power(lx) + _power(ly) + _power(out)) / BYTES_PER_S
    # free range of each side: what the MFMA products need
    dense = union - lx >= 6 and union - ly >= 6 and union - out >= 4
    c += _power(union) / (GEMM_PRODUCTS_PER_S if dense else PRODUCTS_PER_S)
    return c * (BATCH_WEIGHT if batched else 1.0)


def analyse(tree, tables, esize, regroup=True):
    """(post-order FNode list, number of variables no remaining leaf holds -- each doubles the
    count) of a plan, or None when no leaf would remain, or none of those that slicing changes."""
    # the tree's nodes, children before parents
    flat, inner, todo = [], tree.context.nodes, [tree.node_id]
    while todo:  # (each after what is to its right, then turned round)
        t = inner[todo.pop()]
        flat.append(t)
        if not t.is_leaf:
            todo += (t.left, t.right)
    flat.reverse()
    if flat[-1].free_edges:
        raise ValueError("the tree's root has free edges; only full contractions are supported")
    leaves = [(i, tables[n.tensor_index], n.free_edges) for i, n in enumerate(flat) if n.is_leaf]
    root = {}

    def find(e):
        while root.setdefault(e, e) != e:
            root[e] = e = root[root[e]]
        return e

    for i, t, free in leaves:
        if t.rank != len(free):
            raise ValueError("leaf %d: table rank %d != tree rank %d" % (flat[i].tensor_index, t.rank, len(free)))
        if t.copy is not None:
            for e in free:
                root[find(e)] = find(free[0])

    # leaves: variable -> offset mask in the leaf's own table
    offs, weights, hosts = {}, [], []
    seen, sliced, changes = set(), {}, False
    for i, t, free in leaves:
        off, bit = {}, 1 << len(free)
        for e in free:
            bit >>= 1
            v = find(e)
            off[v] = off.get(v, 0) | bit
        seen.update(off)
        changes = changes or t.batched
        if t.copy is not None and t.copy[2] and t.copy[0] == 1 and t.copy[1] == 1:
            continue  # a vector of ones
        offs[i] = off
        sliced[i] = t.batched
        (weights if len(off) <= 1 else hosts).append(i)
    if changes and not any(sliced.values()):
        return None  # every slice counts, though what is left is the same in all of them
    # weight vectors (and scalars) multiply one leaf that holds their variable: an unsliced
    # one where possible, so that the product is not repeated per slice
    attach, placed = {}, set()
    by_var, best = {}, {}  # leaves by variable; the one taken, by variable (None: any) and slicing
    for h in hosts:
        for v in offs[h]:
            by_var.setdefault(v, []).append(h)
    for w in weights:
        v = next(iter(offs[w]), None)
        cand = hosts if v is None else by_var.get(v)
        if cand:
            key = v, sliced[w]
            if key not in best:
                best[key] = min(cand, key=lambda i: (sliced[i] != sliced[w], len(offs[i]), i))
            attach.setdefault(best[key], []).append(w)
            placed.add(w)

    total = {}
    for off in offs.values():
        for v in off:
            total[v] = total.get(v, 0) + 1
    missing = len(seen) - len(total)

    def join(left, right):
        m = dict(left.open)
        for v, c in right.open.items():
            m[v] = m.get(v, 0) + c
        batched = left.batched or right.batched
        union = len(m)
        out = {v: c for v, c in m.items() if c != total[v]}
        return _T(None, out, left, right, batched, union, _join_cost(left, right, union, len(out), batched, esize))

    def leaf(i):
        return _T(i, {v: 1 for v in offs[i]}, batched=sliced[i])

    def absorb(left, right):
        """Their join; where one operand is a large tensor's join with a small one, the small ones
        are joined first if that costs less."""
        t = join(left, right)
        while regroup:
            big, small = (t.left, t.right) if len(t.left.open) >= len(t.right.open) else (t.right, t.left)
            if big.leaf is not None or len(small.open) > SMALL_RANK:
                break
            ib, ism = (big.left, big.right) if len(big.left.open) >= len(big.right.open) else (big.right, big.left)
            if len(ib.open) < BIG_RANK or len(ism.open) > SMALL_RANK:
                break
            m = join(ism, small)
            if len(m.open) > SMALL_RANK:
                break
            nt = join(ib, m)
            if nt.cost + m.cost >= t.cost + big.cost:
                break
            t = nt
        return t

    stack = []
    for i, n in enumerate(flat):
        if n.is_leaf:
            if i not in offs or i in placed:
                stack.append(None)
                continue
            t = leaf(i)
            for w in sorted(attach.get(i, []), key=lambda i: (sliced[i], i)):
                t = absorb(t, leaf(w))
            stack.append(t)
            continue
        right, left = stack.pop(), stack.pop()
        if left is None or right is None:
            stack.append(left or right)
            continue
        stack.append(absorb(left, right))
    top = stack[0]
    if top is None:
        return None

    # post-order nodes; a lone leaf is summed by a join with the constant one (no right child)
    nodes, index, todo = [], {}, [(top, False)]
    while todo:
        t, expanded = todo.pop()
        if t.leaf is None and not expanded:
            todo += [(t, True), (t.right, False), (t.left, False)]
            continue
        n = FNode(len(nodes))
        n.is_leaf = t.leaf is not None
        n.batched = t.batched
        n.left = n.right = -1
        if n.is_leaf:
            n.tensor = flat[t.leaf].tensor_index
            n.rank = len(flat[t.leaf].free_edges)
            n.off = offs[t.leaf]
        else:
            n.left, n.right = index[id(t.left)], index[id(t.right)]
            nodes[n.left].parent = nodes[n.right].parent = n.idx
            n.rank = len(t.open)
        n.order = list(t.open)
        index[id(t)] = n.idx
        nodes.append(n)
    if nodes[-1].is_leaf:
        leaf_node = nodes[-1]
        n = FNode(len(nodes))
        n.is_leaf, n.batched, n.left, n.right, n.rank, n.order = False, leaf_node.batched, leaf_node.idx, -1, 0, []
        leaf_node.parent = n.idx
        nodes.append(n)
    # the plan's one bit order: variables summed later are lower bits, of these the ones that
    # the smaller operands of the larger joins hold less (a wave's loads of such an operand
    # take fewer lines)
    when, weight = {}, {}
    for n in nodes:
        if n.is_leaf:
            continue
        kept = set(n.order)
        held = set(nodes[n.left].order)
        if n.right >= 0:
            held |= set(nodes[n.right].order)
        n.ksum = held - kept
        for v in n.ksum:
            when[v] = n.idx
        if n.right >= 0:
            for v in min(nodes[n.left].order, nodes[n.right].order, key=len):
                weight[v] = weight.get(v, 0.0) + _power(len(held))
    place = {v: i for i, v in enumerate(sorted(when, key=lambda v: (-when[v], weight.get(v, 0.0), v)))}
    for n in nodes:
        n.order.sort(key=place.__getitem__)
        n.order0 = n.order
    return nodes, missing


def _reordered(n, order):
    n.order = order
    n.off = {v: 1 << i for i, v in enumerate(order)}


def _canonical(node, want):
    """True when a stored tensor's bits are the variables ``want`` in order."""
    return node.rank == len(want) and all(node.off.get(v) == 1 << i for i, v in enumerate(want))


def _vec_form(xoff, yoff, xrank, yrank, out, off, ksum, nb, launch_bound):
    """The 16-byte form of a join that streams the operand of offsets ``xoff``, or None."""
    yonly = [v for v in out if v not in xoff]
    reg = yonly[:MAX_REG_BITS]
    body = [v for v in out if v not in reg] if reg else out
    s = len(ksum)
    if len(body) < 10 or xoff.get(body[0]) != 1 or xoff.get(body[1]) != 2 or off[body[0]] != 1 or \
            off[body[1]] != 2 or xrank < 2 or (int(math.log2(nb)) + len(body) < 18 and s > 4) or \
            len(body) + s + len(reg) > _lib.FOLD_BITS:
        return None
    # shared range in the streamed operand's memory order, lowest first
    ks = sorted(ksum, key=lambda v: (xoff.get(v, 1 << 40), yoff.get(v, 0), v))
    y0, y1 = yoff.get(body[0], 0), yoff.get(body[1], 0)
    if not y0 or not y1:
        ym = 3 if y0 else 4 if y1 else 0
        if not ym and yrank >= 2 and [yoff.get(v) for v in reg[:2]] == [1, 2]:
            ym = 5
    else:
        ym = 1 if (y0, y1) == (1, 2) and yrank >= 2 else 2
    if launch_bound:  # fewer launches a step, the forms that the others are cases of: 890 -> 868 us (96 instances)
        ym = {3: 2, 4: 2, 5: 0}.get(ym, ym)
    ntile = len(body) - 10
    return dict(kind="fold", variant=_lib.TO_FOLD_VEC | ym << 4 | len(reg), bits=body + ks + reg, fy=len(yonly),
                roles=(10, 0, ntile, s, 0, len(reg)), nblocks=int(min(nb << ntile, MAX_VEC_BLOCKS)), lsplit=0,
                vec=True, yc=1 << len(reg))


def choose(n, nodes, W, esize, launch_bound=False):
    """Kernel form and launch shape of one folded join for W slices (``n.geom``).  A dense
    join also fixes its result's bit order ([kept shared][X][Y]).  ``launch_bound`` (the
    many-instance batch): every product in the 64x64 form, so that those of a step share a
    launch."""
    A = nodes[n.left]
    B = nodes[n.right] if n.right >= 0 else None
    nb = W if n.batched else 1
    if max(t.rank for t in (A, B, n) if t is not None) > OFFSET_BITS:
        raise TooWide("folded join of a tensor of more than 2^%d entries" % OFFSET_BITS)
    _reordered(n, list(n.want or n.order0))
    if B is None:
        X, Y = A, None
    else:
        X, Y = (A, B) if (A.rank, A.batched) >= (B.rank, B.batched) else (B, A)
    xoff = X.off
    yoff = Y.off if Y is not None else {}
    # shared range in X's memory order, lowest first
    ks = sorted(n.ksum, key=lambda v: (xoff.get(v, 1 << 40), yoff.get(v, 0), v)) if len(n.ksum) > 1 else list(n.ksum)
    s = len(ks)
    if Y is not None and n.rank >= 2 * schedule.GEMM_MIN_FREE and all(v in xoff and v in yoff for v in ks):
        kept = [v for v in n.order if v in xoff and v in yoff]
        xo = [v for v in n.order if v in xoff and v not in yoff]
        yo = [v for v in n.order if v in yoff and v not in xoff]
        plain = X.rank == len(xoff) and Y.rank == len(yoff)
        if len(xo) >= schedule.GEMM_MIN_FREE and len(yo) >= schedule.GEMM_MIN_FREE and \
                s >= schedule.GEMM_MIN_SHARED and plain and \
                (not kept or nb == 1 or (X.batched and Y.batched)):
            if len(yo) > len(xo):
                X, Y, xo, yo = Y, X, yo, xo
            h = len(kept)
            _reordered(n, yo + xo + kept)
            g = dict(fx=len(xo), fy=len(yo), s=s, shf=len(yo), shy=0, xf=list(range(s, s + len(xo))),
                     xs=list(range(s)), yf=list(range(s, s + len(yo))), ys=list(range(s)), x_is_left=X is A)
            v = schedule.choose_variant(g, nb << h, esize, launch_bound=launch_bound)
            if h and v.get("lsplit"):  # the finishing launch has one record per batch item
                del v["lsplit"], v["nsplit"], v["nout"], v["fin_blocks"]
                v["nblocks"] = int(min((nb << h) << (len(xo) + len(yo) - 12), schedule.MAX_GEMM_BLOCKS))
            want_x, want_y = ks + xo + kept, ks + yo + kept
            for t, want in ((X, want_x), (Y, want_y)):
                if not t.is_leaf and not _canonical(t, want) and t.geom["var"]["kind"] == "fold" and \
                        t.rank <= TREE_RANK and (W if t.batched else 1) << t.rank <= WANT_ENTRIES:
                    t.want = want
                    choose(t, nodes, W, esize, launch_bound)
            v.update(perm_x=not _canonical(X, want_x), perm_y=not _canonical(Y, want_y), hlog=h, want_x=want_x,
                     want_y=want_y)
            g.update(var=v, X=X.idx, Y=Y.idx)
            n.geom = g
            return
    out = n.order
    nc = len(out)
    lognb = int(math.log2(nb))
    # the 16-byte form, streaming the operand that has the outputs' two lowest variables as its
    # own: the larger one, else the other (2^16 by 2^16 over 2^3 to 2^20, 4096 slices: 6.4 ms as
    # a register tile with 4-byte stores, 5.7 here)
    for x, y in ((X, Y), (Y, X)) if Y is not None and nc >= 10 else ():
        v = _vec_form(x.off, y.off, x.rank, y.rank, out, n.off, n.ksum, nb, launch_bound)
        if v is not None:
            n.geom = dict(fx=nc - v["fy"], fy=v["fy"], s=s, X=x.idx, Y=y.idx, var=v)
            return
    yonly = [v for v in out if v not in xoff]
    g = dict(fx=nc - len(yonly), fy=len(yonly), s=s, X=X.idx, Y=Y.idx if Y is not None else -1)
    # register tile: outputs enough to fill the chip without the tile's bits
    xonly = [v for v in out if v not in yoff]
    for na, nbits in REG_TILES if Y is not None and nc >= 10 else ():
        if len(xonly) < na or len(yonly) < nbits or nc - na - nbits < 8 or lognb + nc - na - nbits < REG_MIN_LOG:
            continue
        # the tile's variables: the highest bits of the result, so that the lanes keep low ones
        reg = (xonly[len(xonly) - na:] if na else []) + (yonly[len(yonly) - nbits:] if nbits else [])
        body = [v for v in out if v not in reg]
        ntile = len(body) - 8
        g["var"] = dict(kind="fold", variant=_lib.TO_FOLD_REG | na << 4 | nbits, bits=body + ks + reg,
                        roles=(8, 0, ntile, s, 0, na + nbits), nblocks=int(min(nb << ntile, MAX_ANY_BLOCKS)), lsplit=0,
                        vec=False, yc=1)
        if len(g["var"]["bits"]) <= _lib.FOLD_BITS:
            n.geom = g
            return
    # general form: thread bits go to outputs, then to the shared range while the launch
    # would have few threads; long shared ranges with few outputs are split over blocks
    dot = s >= DOT_MIN_SHARED and nc <= 6 and all((xoff.get(v), yoff.get(v)) == (o, o) for v, o in zip(ks, (1, 2))) \
        and X.rank >= 2 and Y.rank >= 2
    if dot:  # its four consecutive shared indices go with one load
        ks = ks[2:]
        s -= 2
    lk = 0
    if lognb + nc < ANY_MIN_THREADS_LOG and s > 0:
        lk = min(s, 8, max(8 - nc, min(s - 3, ANY_MIN_THREADS_LOG - lognb - nc)))
        lk = max(lk, 0)
    lo = min(nc, 8 - lk)
    rest = s - lk
    lsplit = 0
    if rest > 6:
        lsplit = max(0, min(rest - 4, ANY_MIN_THREADS_LOG + 3 - lognb - nc - lk))
    ntile = nc - lo
    pad = [None] * (8 - lo - lk)
    g["var"] = dict(kind="fold", variant=_lib.TO_FOLD_DOT if dot else _lib.TO_FOLD_ANY,
                    bits=out[:lo] + ks[:lk] + pad + out[lo:] + ks[lk:],
                    roles=(lo, lk, ntile, rest - lsplit, lsplit, 0),
                    nblocks=int(min(nb << (ntile + lsplit), MAX_ANY_BLOCKS)), lsplit=lsplit, nout=nb << nc,
                    nsplit=1 << lsplit, vec=False, yc=1)
    if len(g["var"]["bits"]) > _lib.FOLD_BITS:
        raise TooWide("folded join over more than %d variables" % _lib.FOLD_BITS)
    n.geom = g


def choose_all(nodes, W, esize, launch_bound=False):
    nodes[-1].layout = None
    if esize == 4 and len(nodes) > EXPONENT_NODES:
        raise TooWide("more than %d nodes" % EXPONENT_NODES)
    for n in nodes:
        n.want = None
    for n in nodes:
        if not n.is_leaf:
            choose(n, nodes, W, esize, launch_bound)
    if not launch_bound and not nodes[-1].is_leaf:
        _fuse(nodes[-1], nodes, W)


def _fuse(n, nodes, W):
    """The dot product at the root with the joins that make its operands, or one of them, run
    inside it (TO_OP_FOLD_PAIR): each stores and reads back a large tensor otherwise (the
    2^20-entry operands of 4096 slices: 7.4 + 7.3 ms for the joins and 5.6 for the dot).  Only
    joins too large for a program, that sum at most two variables: their large operand is then
    read about once."""
    if n.geom["var"].get("variant") != _lib.TO_FOLD_DOT or n.rank or n.left < 0:
        return

    def side(c):
        f = nodes[c]
        if f.is_leaf or f.right < 0 or f.batched != n.batched or f.geom["var"]["kind"] != "fold" or \
                f.rank <= TREE_RANK or len(f.ksum) > 2:
            return None
        x, y = nodes[f.geom["X"]], nodes[f.geom["Y"]]
        return (x, y, sorted(f.ksum), f) if x.rank >= y.rank else (y, x, sorted(f.ksum), f)

    plain = [(nodes[c], None, [], None) for c in (n.geom["X"], n.geom["Y"])]
    inner = [side(c) for c in (n.geom["X"], n.geom["Y"])]
    for pair in ((inner[0], inner[1]), (inner[0], plain[1]), (inner[1], plain[0])):
        if None in pair:
            continue
        a, b = sorted(pair, key=lambda p: -len(p[2]))
        xa, xb = a[0].off, b[0].off
        order = sorted(n.ksum, key=lambda v: (xa.get(v, 1 << 40), xb.get(v, 1 << 40), v))
        body = [v for v in order if v in xa]
        reg = [v for v in order if v not in xa]
        # the variables only X0 has change fastest (X1's entries come again from a cache)
        wide = [v for v in body if v in xb][:10]
        body = wide + [v for v in body if v not in xb] + [v for v in body if v in xb and v not in wide]
        bits = body + reg + a[2] + b[2]
        if len(body) < 10 or len(reg) > 4 or len(bits) > _lib.FOLD_BITS or \
                any(x.get(body[0]) != 1 or x.get(body[1]) != 2 for x in (xa, xb)):
            continue

        lows = any(y is not None and (v in y.off) for v in body[:2] for y in (a[1], b[1]))
        nb = W if n.batched else 1
        lsplit = max(0, min(len(body) - 10, PAIR_MIN_BLOCKS_LOG - int(math.log2(nb))))
        reads = [t.idx for s in (a, b) for t in s[:2] if t is not None]
        n.geom.update(reads=reads, var=dict(
            kind="pair", variant=len(a[2]) << 4 | len(b[2]) | (0 if lows else _lib.TO_PAIR_ONE), sides=(a, b), bits=bits,
            nreg=len(reg),
            nloop=len(body) - 10 - lsplit, lsplit=lsplit, nsplit=1 << lsplit, nout=nb,
            nblocks=int(min(nb << lsplit, MAX_ANY_BLOCKS))))
        for s in (a, b):
            if s[3] is not None:
                s[3].geom["var"] = dict(kind="fused")
        return


def _reads(n):
    """The tensors a join reads (of a fused one, those its parts read)."""
    return n.geom.get("reads") or [c for c in (n.left, n.right) if c >= 0]


def _fused(n):
    return not n.is_leaf and n.geom["var"]["kind"] == "fused"


def _scratch(arena, n, nodes, nb, esize, table):
    """Scratch a join needs while it runs: split sums, permuted operands of a product."""
    v = n.geom["var"]
    blocks = {}
    if v.get("lsplit"):
        blocks["partial"] = arena.alloc(v["nout"] * v["nsplit"] * 8)
    if v["kind"] == "gemm":
        for key, i in (("perm_x", n.geom["X"]), ("perm_y", n.geom["Y"])):
            if v[key]:
                blocks[key] = arena.alloc((nb if nodes[i].batched else 1) * (1 << nodes[i].rank) * esize)
    table[n.idx] = blocks
    return list(blocks.values())


class TreeProgram:
    """A connected part of the tree, of small joins, that a block runs for one slice: its
    joins by level as (node, operands), what each sums, the LDS element offsets and record
    slots of their results (the root's goes to the arena) and the LDS bytes."""

    __slots__ = ("root", "members", "levels", "sums", "at", "slot", "lds", "batched", "outside")


def _merge(nodes, members):
    """Operands and summed variables of the joins of a program after small joins are merged
    into the products they feed ({join: operands}, {join: variables})."""
    ops, sums, level = {}, {}, {}
    for i in sorted(members):
        n = nodes[i]
        mine, ks = [c for c in (n.left, n.right) if c >= 0], set(n.ksum)
        while True:
            best = None
            for c in mine:
                if c not in ops or len(mine) - 1 + len(ops[c]) > 4 or len(ks) + len(sums[c]) > MERGE_LOOP \
                        or n.rank > 6:
                    continue
                if best is None or level[c] > level[best]:
                    best = c
            if best is None:
                break
            mine = [c for c in mine if c != best] + ops.pop(best)
            ks |= sums.pop(best)
        ops[i], sums[i] = mine, ks
        level[i] = 1 + max((level[c] for c in mine if c in ops), default=0)
    return ops, sums, level


def _program(nodes, root, stage, esize, scaled):
    p = TreeProgram()
    p.root, p.batched = root, nodes[root].batched
    todo, p.members = [root], set()
    while todo:
        i = todo.pop()
        p.members.add(i)
        todo += [c for c in (nodes[i].left, nodes[i].right) if stage.get(c) == stage[root]]
    ops, p.sums, level = _merge(nodes, p.members)
    p.levels = [[] for _ in range(level[root])]
    for i in ops:
        p.levels[level[i] - 1].append((i, ops[i]))
    arena, p.at, live = schedule._Arena(align=16), {}, {}
    for lv in p.levels:
        for i, _ in lv:
            if i != root:
                live[i] = arena.alloc(esize << nodes[i].rank)
                p.at[i] = live[i][0] // esize
        for _, mine in lv:
            for c in mine:
                if c in live:
                    arena.release(live.pop(c))
    p.slot = {i: k for k, i in enumerate(p.at)}
    p.lds = arena.peak + ((8 * len(p.slot) + 15) & ~15 if scaled else 0)
    # tensors of the same phase that other launches make
    p.outside = [c for _, mine in ((i, m) for lv in p.levels for i, m in lv) for c in mine
                 if c not in p.at and not nodes[c].is_leaf and nodes[c].batched == p.batched]
    return p


def tree_programs(nodes, W, esize, scaled, lds=None):
    """The programs of a plan whose joins carry their forms: connected parts of small joins of
    one phase whose intermediates fit ``lds`` bytes, of at most TREE_PRODUCTS products."""
    # a small join's stage: its phase and the number of large joins -- and of places where a
    # program ends because it may hold no more -- on the longest path below it; programs are the
    # connected joins of one stage, so none waits for more than it reads
    joins = [n for n in nodes if not n.is_leaf]
    at = {n.idx: k for k, n in enumerate(joins)}
    stage, depth = {}, {}
    size = {}  # joins of the program that ends at a small join
    sure = {}  # ... and how many of them one join below it has been seen to hold
    full = set()  # joins that do not fit one program with what is below them

    def fits(i):
        p = _program(nodes, i, stage, esize, scaled)
        ok = p.lds <= (lds or (TREE_LDS_MANY if p.batched and W >= TREE_MANY else TREE_LDS)) and \
            sum(map(len, p.levels)) <= TREE_PRODUCTS
        if ok:
            sure[i] = size[i]
        return p if ok else None

    def first_full(i):
        """The first join of the program ending at ``i``, which does not fit, that is too much."""
        todo, members = [i], []
        while todo:
            members.append(todo.pop())
            todo += [c for c in (nodes[members[-1]].left, nodes[members[-1]].right) if stage.get(c) == stage[i]]
        members.sort()
        lo, hi = 0, len(members)  # of the first lo joins every program fits, of the first hi one does not
        while hi - lo > 1:
            mid = (lo + hi) // 2
            tops = [m for m in members[:mid] if nodes[m].parent > members[mid - 1]]
            if all(sure[m] == size[m] or fits(m) for m in tops):
                lo = mid
            else:
                hi = mid
        return members[hi - 1]

    k, out = 0, []
    while True:
        while k < len(joins):
            n = joins[k]
            i, cut = n.idx, n.idx in full
            below, far, deep = [], False, 0
            for c in (n.left, n.right):
                if c >= 0:
                    near = nodes[c].batched == n.batched
                    # a block reads a large tensor of another launch at the latency of L2: fewer products
                    far = far or nodes[c].rank > TREE_FAR_RANK and (cut or not near or c not in stage)
                    if near and c in depth:
                        below.append(c)
                        deep = max(deep, depth[c])
            small = n.geom["var"]["kind"] == "fold" and n.rank <= TREE_RANK and \
                len(n.ksum) + n.rank <= (TREE_FAR_BITS if far else TREE_BITS)
            if cut or not small:
                deep += 1
            depth[i] = deep
            k += 1
            if not small:
                stage.pop(i, None)
                continue
            stage[i] = mine = (n.batched, deep)
            held, known = 1, 1
            for c in below:
                if stage.get(c) == mine:
                    held += size[c]
                    known = max(known, sure[c])
            size[i], sure[i] = held, known
            # (long ones are checked where they have doubled, so that a join is looked at a few
            # times in all; the others where they end)
            if held > TREE_LONG and held > 2 * known and fits(i) is None:
                j = first_full(i)
                full.add(j)
                k = at[j]
        out, again = [], []
        for i in stage:
            if stage.get(nodes[i].parent) != stage[i]:
                p = fits(i)
                if p is None:
                    again.append(first_full(i))
                elif size[i] > 1 or len(nodes[i].ksum) + nodes[i].rank <= TREE_LONE_BITS:
                    out.append(p)
        if not again:
            return sorted(out, key=lambda p: p.root)
        full.update(again)
        k = min(at[j] for j in again)


def _tree_task(n, ksum, operands):
    """(lo, lk, nloop, nchunk), variables in bit order, of a join inside a program.  Short
    sums are walked by one lane; longer ones are shared by the lanes the outputs leave."""
    def key(v):
        return tuple(t.off.get(v, 1 << 40) for t in operands) + (v,)

    ks = sorted(ksum, key=key) if len(ksum) > 1 else list(ksum)
    nc, s = n.rank, len(ks)
    lo = min(nc, 6)
    lk = max(0, min(s - 2, 6 - lo))
    bits = n.order[:lo] + ks[:lk] + [None] * (6 - lo - lk) + n.order[lo:] + ks[lk:]
    return (lo, lk, s - lk, nc - lo), bits


def tree_words(p, nodes, waves, rec_index, one):
    """(uint32 joins [n, 128], uint32 task streams [waves, ntask]) of a program.  ``one``:
    (address, record index) of the stored 1.0."""
    words = np.zeros((sum(map(len, p.levels)), _lib.TO_TREE_WORDS), dtype=np.uint32)
    if len(words) > TREE_PRODUCTS:
        raise ValueError("a program of %d products" % len(words))
    streams = [[] for _ in range(waves)]
    k = 0
    for lv in p.levels:
        costs, tasks = [], []
        for i, mine in lv:
            n = nodes[i]
            # the walk of two operands takes the one with more variables first
            mine = sorted(mine, key=lambda c: -len(nodes[c].order))
            if len(mine) == 1:
                mine = mine + [-1]
            (lo, lk, nloop, nchunk), bits = _tree_task(n, p.sums[i], [nodes[c] for c in mine if c >= 0])
            row = [0] * 128
            head = lo | lk << 4 | nloop << 8 | nchunk << 12 | (len(mine) - 1) << 16
            for j, t in list(enumerate(mine)) + [(4, i)]:
                if t in p.at:
                    head |= 1 << (20 + j)
                    row[1 + 2 * j], row[16 + j] = p.at[t], p.slot[t]
                else:
                    addr, rec, stride, advances = (one[0], one[1], 0, 0) if t < 0 else (
                        nodes[t].ptr, rec_index(nodes[t]), nodes[t].bstride if p.batched else 0,
                        nodes[t].rec_stride if p.batched else 0)
                    row[1 + 2 * j], row[2 + 2 * j] = addr & 0xffffffff, addr >> 32
                    row[11 + j], row[16 + j] = stride, rec
                    head |= (1 << (25 + j)) if advances else 0
                off = nodes[t].off if t >= 0 else {}
                at = 64 + 16 * j if j < 4 else 32
                for b, v in enumerate(bits):
                    if v is not None:
                        row[at + b] = off.get(v, 0)
            row[0] = head
            words[k, :128] = row
            # rough wave cycles: setting up, then per chunk its loads
            costs.append((300, (1 << nchunk) * (100 + (30 * len(mine) << nloop) // 2), nchunk, k))
            k += 1
        share = sum(c[1] for c in costs) / waves
        for setup, work, nchunk, j in costs:
            lstep = 0
            while lstep < nchunk and (1 << lstep) < waves and work / (1 << lstep) > max(share, 2 * setup):
                lstep += 1
            tasks += [(setup + work / (1 << lstep), j | c << 16 | lstep << 23) for c in range(1 << lstep)]
        tasks.sort(key=lambda t: -t[0])
        load, mine = [0.0] * waves, [[] for _ in range(waves)]
        for cost, word in tasks:
            w = load.index(min(load))
            load[w] += cost
            mine[w].append(word)
        rounds = max(len(m) for m in mine)
        for w in range(waves):
            m = mine[w] + [_lib.TO_TREE_IDLE] * (rounds - len(mine[w]))
            m[-1] |= _lib.TO_TREE_MEET
            streams[w] += m
    # every lane's offset: the sum of the entries of its bits, for operands 0-3 and the result
    words[:, 128:] = (words[:, _LANE_ENTRIES].reshape(-1, 5, 6) @ _LANE_BITS).reshape(-1, 5 * 64)
    return words, np.array(streams, dtype=np.uint32)


def phase_groups(nodes, batched, order, programs):
    """Groups of one phase in execution order, each (programs, joins) that may run together.
    ``order`` "level": every unit (a program, or a join outside all of them) one level above
    the highest of what it reads; "post": the programs that read nothing of the phase first,
    then unit by unit."""
    mine = [p for p in programs if p.batched == batched]
    unit = {i: p for p in mine for i in p.members}
    level, out = {}, []
    first = []
    for n in nodes:
        if n.is_leaf or n.batched != batched or _fused(n):
            continue
        p = unit.get(n.idx)
        if p is not None and p.root != n.idx:
            continue
        lv = 1 + max((level.get(c, 0) for c in (p.outside if p is not None else _reads(n))), default=0)
        level[n.idx] = lv
        if order == "level":
            while len(out) < lv:
                out.append(([], []))
            (out[lv - 1][0] if p is not None else out[lv - 1][1]).append(p if p is not None else n.idx)
        elif p is not None and lv == 1:
            first.append(p)
        else:
            out.append(([p], []) if p is not None else ([], [n.idx]))
    return ([(first, [])] if first else []) + out


def plan_memory(nodes, W, esize, order, programs=()):
    """(arena peak, scratch placements), as ``schedule.plan_memory``; what a program keeps in
    LDS has no place in the arena."""
    arena = schedule._Arena()
    scratch = {}

    def run(group, nb, release):
        temps = []
        for i in [p.root for p in group[0]] + group[1]:
            nodes[i].buf = arena.alloc(nb * (1 << nodes[i].rank) * esize)
        for i in group[1]:
            temps += _scratch(arena, nodes[i], nodes, nb, esize, scratch)
        for blk in temps:
            arena.release(blk)
        read = [c for p in group[0] for lv in p.levels for _, mine in lv for c in mine if c not in p.at]
        read += [c for i in group[1] for c in _reads(nodes[i])]
        for c in read:
            if release(nodes[c]):
                arena.release(nodes[c].buf)

    for grp in phase_groups(nodes, False, order, programs):
        run(grp, 1, lambda c: not c.is_leaf and not c.batched)
    for n in nodes:
        if n.is_leaf and n.batched:
            n.buf = arena.alloc(W * (1 << n.rank) * esize)
    for grp in phase_groups(nodes, True, order, programs):
        run(grp, W, lambda c: c.batched)
    return arena.peak, scratch


def choose_order(nodes, W, esize, programs=()):
    """(order, arena peak, scratch placements): level launches unless they take far more
    memory."""
    level, scratch = plan_memory(nodes, W, esize, "level", programs)
    if level <= LEVEL_FREE_BYTES:
        return "level", level, scratch
    post, scratch = plan_memory(nodes, W, esize, "post", programs)
    if level <= schedule.LEVEL_PEAK_FACTOR * post:
        return "level", *plan_memory(nodes, W, esize, "level", programs)
    return "post", post, scratch


def lay_out(nodes, W, esize, group_levels=True):
    """Forms, programs and memory plan of a folded plan for W slices: (programs, order, arena
    peak, scratch placements)."""
    choose_all(nodes, W, esize)
    if not group_levels:
        return [], "post", *plan_memory(nodes, W, esize, "post", [])
    programs = tree_programs(nodes, W, esize, esize == 4)
    return programs, *choose_order(nodes, W, esize, programs)


def peak_bytes(nodes, W, esize):
    """Arena bytes for W slices; the layout stays with the plan for ``compile_program``."""
    layout = lay_out(nodes, W, esize)
    nodes[-1].layout = (W, esize), layout
    return layout[2]


def join_records(n, nodes, W, esize, scaled, abase, scratch, recp, one, launch_bound=False):
    """Descriptor records of one join in execution order, as ``schedule.join_records``:
    [(kind, op, variant, lds, descriptor, blocks)]; ``one``: (address, record address) of a
    stored 1.0, the second operand of a lone leaf's sum; ``launch_bound`` (the many-instance
    batch): permutes in one form, so that those of a step share a launch."""
    g, v = n.geom, n.geom["var"]
    nb = W if n.batched else 1
    X = nodes[g["X"]]
    Y = nodes[g["Y"]] if g["Y"] >= 0 else None
    out = []
    if v["kind"] == "gemm":
        ops = []
        for key, op, want in (("perm_x", X, v["want_x"]), ("perm_y", Y, v["want_y"])):
            stride = (1 << op.rank) if (n.batched and op.batched) else 0
            if v[key]:
                dst = abase + scratch[key][0]
                out_pos = [0] * op.rank
                for i, var in enumerate(want):
                    out_pos[op.off[var].bit_length() - 1] = i
                pd, grid, lds, pvar = schedule.perm_desc(op.ptr, dst, op.rank, out_pos,
                                                         W if (n.batched and op.batched) else 1, 1 << op.rank, esize,
                                                         not launch_bound)
                out.append(("permute", _lib.TO_OP_PERMUTE, pvar, lds, pd, grid))
                ops.append((dst, stride))
            else:
                ops.append((op.ptr, stride))
        gd = _lib.GemmDesc()
        h = v["hlog"]
        gd.a, gd.b, gd.c = ops[0][0], ops[1][0], n.ptr
        gd.mlog, gd.nlog, gd.klog = g["fx"], g["fy"], g["s"]
        gd.hlog = h
        gd.ldcm, gd.ldcn = 1 << g["shf"], 1 << g["shy"]
        if scaled:
            gd.as_, gd.bs, gd.cs = recp(X), recp(Y), recp(n)
            gd.asb = X.rec_stride if n.batched else 0
            gd.bsb = Y.rec_stride if n.batched else 0
        gd.block0, gd.nblocks = 0, v["nblocks"]
        # batch items are (slice, kept shared variables); an operand without slices would
        # repeat its 2^h items per slice, which one batch stride cannot say (see ``choose``)
        gd.ab = 1 << (g["fx"] + g["s"]) if (ops[0][1] or h) else 0
        gd.bb = 1 << (g["fy"] + g["s"]) if (ops[1][1] or h) else 0
        gd.cb = 1 << (g["fx"] + g["fy"])
        gd.nbatch = nb << h
        out.append(("gemm", _lib.TO_OP_GEMM, v["tile"], 0, gd, v["nblocks"]))
        if v.get("lsplit"):
            # split K: the parts' partial sums go to scratch, a finishing launch writes C
            f = _lib.JoinDesc()
            f.c, f.cb, f.nsplit = n.ptr, n.bstride, v["nsplit"]
            gd.c = f.partial = abase + scratch["partial"][0]
            gd.lsplit = v["lsplit"]
            f.xs, f.ys, f.cs, f.xsb, f.ysb = gd.as_, gd.bs, gd.cs, gd.asb, gd.bsb
            f.fx, f.fy, f.shf, f.shy, f.nbatch, f.nblocks = g["fx"], g["fy"], g["shf"], 0, nb, v["fin_blocks"]
            out.append(("finish", _lib.TO_OP_JOIN_FINISH, 0, 0, f, f.nblocks))
        return out
    if v["kind"] == "pair":
        return pair_records(n, W, esize, scaled, abase, scratch, recp, one)
    d = FoldDesc()
    yptr, yrec, ystride, yrecs = one[0], one[1], 0, 0
    if Y is not None:
        yptr, yrec = Y.ptr, recp(Y)
        ystride = Y.bstride if n.batched else 0
        yrecs = Y.rec_stride if n.batched else 0
    partial = abase + scratch["partial"][0] if v["lsplit"] else 0
    d.ptrs = (X.ptr, yptr, n.ptr)
    d.strides = (X.bstride if n.batched else 0, ystride, n.bstride)
    d.recs = (recp(X), yrec, recp(n)) if scaled else (0, 0, 0)
    d.rec_strides = (X.rec_stride if n.batched else 0, yrecs)
    d.partial = partial
    d.nbatch, d.block0, d.nblocks, d.roles = nb, 0, v["nblocks"], v["roles"]
    yoff = Y.off if Y is not None else {}
    fill = [0] * (_lib.FOLD_BITS - len(v["bits"]))
    d.bits = [X.off.get(b, 0) for b in v["bits"]] + fill + [yoff.get(b, 0) for b in v["bits"]] + fill \
        + [n.off.get(b, 0) for b in v["bits"]] + fill
    out.append(("fold", _lib.TO_OP_FOLD, v["variant"], 0, d, v["nblocks"]))
    if v["lsplit"]:
        out.append(_finish(n, v, partial, nb, list(zip(d.recs, d.rec_strides)) if scaled else [], d.recs[2]))
    return out


def pair_records(n, W, esize, scaled, abase, scratch, recp, one):
    """Descriptor records of a fused dot product (see ``join_records``)."""
    v = n.geom["var"]
    nb = W if n.batched else 1
    d = _lib.PairDesc(c=n.ptr, cb=n.bstride, cs=recp(n) if scaled else 0, nbatch=nb, nblocks=v["nblocks"],
                      nloop=v["nloop"], lsplit=v["lsplit"], nreg=v["nreg"])
    nbits = len(v["bits"])
    ends = []
    for k, (X, Y, ksum, f) in enumerate(v["sides"]):
        d.x[k], d.xb[k] = X.ptr, X.bstride if n.batched else 0
        d.y[k], d.yb[k] = (Y.ptr, Y.bstride if n.batched else 0) if Y is not None else (one[0], 0)
        d.nk[k] = len(ksum)
        d.bx[k][:nbits] = [X.off.get(b, 0) for b in v["bits"]]
        d.by[k][:nbits] = [Y.off.get(b, 0) if Y is not None else 0 for b in v["bits"]]
        if scaled:
            d.xs[k], d.xsb[k] = recp(X), X.rec_stride if n.batched else 0
            if Y is not None:
                d.ys[k], d.ysb[k] = recp(Y), Y.rec_stride if n.batched else 0
            if f is not None:
                d.rs[k] = recp(f)
            ends.append((recp(f), f.rec_stride if n.batched else 0) if f is not None else (d.xs[k], d.xsb[k]))
    out = [("pair", _lib.TO_OP_FOLD_PAIR, v["variant"], 0, d, v["nblocks"])]
    if v["lsplit"]:
        d.partial = abase + scratch["partial"][0]
        out.append(_finish(n, v, d.partial, nb, ends, d.cs, _lib.TO_FINISH_NORM if scaled else 0))
    return out


def _finish(n, v, partial, nb, ends, crec, norm=0):
    """The record that adds up a join's partial sums; ``ends``: (record, stride) of the two
    operands, whose exponents the result carries (scaled only); ``norm``: TO_FINISH_NORM for a
    sum of products of more than two stored tensors."""
    f = _lib.JoinDesc()
    f.c, f.cb, f.partial, f.nsplit = n.ptr, n.bstride, partial, v["nsplit"]
    if ends:
        (f.xs, f.xsb), (f.ys, f.ysb), f.cs = ends[0], ends[1], crec
    f.fx, f.nbatch = n.rank, nb
    wide = v["nsplit"] >= 32
    f.nblocks = int(min(v["nout"] if wide else -(-v["nout"] // 256), schedule.MAX_STREAM_BLOCKS))
    return "finish", _lib.TO_OP_JOIN_FINISH, norm | wide, 0, f, f.nblocks


def join_traffic(n, nodes, W, esize):
    """Algorithmic (bytes, flops) of one folded join."""
    nb = W if n.batched else 1
    total = (1 << n.rank) * nb
    held = set(n.ksum) | set(n.order)
    for c in (n.left, n.right):
        if c >= 0:
            total += (1 << len(nodes[c].order)) * (nb if nodes[c].batched else 1)
    return total * esize, 2 * nb << len(held)


def block_cost(st):
    if isinstance(st, FoldDesc):
        lo, lk, ntile, nloop, lsplit, nreg = st.roles
        return (1 << (nloop + nreg)) * max(1, (st.nbatch << (ntile + lsplit)) // max(1, st.nblocks))
    return schedule.block_cost(st)


def compile_program(folded, tables, num_groups, entry_type, W, device_alloc, group_levels=True, host_alloc=None):
    """Build a ``schedule.Program`` of a folded plan (``folded``: what ``analyse`` returned)
    for W slices.  The program starts its own sum (TO_OP_ROOT_REDUCE, variant 1), so a run is
    its prologue and waves alone; with ``host_alloc`` (host memory that the device writes)
    the sum also lands there."""
    nodes, missing = folded
    esize = 8 if entry_type == _lib.TO_F64 else 4
    scaled = entry_type == _lib.TO_F32S
    prog = schedule.Program()
    prog.nbatch, prog.nodes = W, nodes
    # (the layout that the batch size was accepted with, if the joins' forms are still its own)
    known, nodes[-1].layout = nodes[-1].layout, None
    if group_levels and known is not None and known[0] == (W, esize):
        programs, order, peak, scratch = known[1]
    else:
        programs, order, peak, scratch = lay_out(nodes, W, esize, group_levels)
    prog.programs = programs
    in_lds = {i for p in programs for i in p.members if i != p.root}
    prog.arena_bytes, prog.order = peak, order

    image = schedule.leaf_image(nodes, tables, num_groups, scaled, np.float64 if esize == 8 else np.float32)
    mant, exp = image.factor
    prog.leaf_factor = (mant, exp + missing)  # a variable no leaf holds counts twice
    one = len(image.host)  # a stored 1.0, after the tables
    image.host = np.concatenate([image.host, np.ones(1, image.host.dtype)])

    # scale records: [constant leaves, the constant one][constant joins][wave tensors]
    nrec, rec_init = 0, []
    if scaled:
        for n in nodes:
            if n.is_leaf and not n.batched:
                n.rec, n.rec_stride = nrec, 0
                rec_init.append((nrec, image.exp0[n.tensor]))
                nrec += 1
        one_rec = nrec
        rec_init.append((nrec, 0))
        nrec += 1
        pro_rec0 = nrec
        for n in nodes:
            if not n.is_leaf and not n.batched and n.idx not in in_lds:
                n.rec, n.rec_stride = nrec, 0
                nrec += 1
        wave_rec0 = nrec
        for leaves in (True, False):  # the gather writes the leaves' records, the rest is cleared
            for n in nodes:
                if n.batched and n.is_leaf == leaves and n.idx not in in_lds:
                    n.rec, n.rec_stride = nrec, 1
                    nrec += W
            if leaves:
                clear_rec0 = nrec
        prog.rec_ranges = (pro_rec0, wave_rec0, nrec)

    prog.table = device_alloc(image.host.nbytes)
    prog.coef = device_alloc(image.coef_host.nbytes)
    prog.arena = device_alloc(max(ALIGN, peak))
    prog.recs = device_alloc(max(1, nrec) * 16)
    prog.params = device_alloc(4 * 8)
    prog.accum = device_alloc(32)
    prog.host_accum = host_alloc(32) if host_alloc is not None else None
    prog.table_host, prog.coef_host, prog.rec_init = image.host, image.coef_host, rec_init
    tbase, abase, rbase = prog.table.data_ptr(), prog.arena.data_ptr(), prog.recs.data_ptr()
    wave_params = prog.params.data_ptr()
    one_at = (tbase + one * esize, rbase + one_rec * 16 if scaled else 0)
    for n in nodes:
        if n.idx in in_lds or _fused(n):
            continue
        if n.is_leaf and not n.batched:
            n.ptr, n.bstride = tbase + image.off[n.tensor] * esize, 0
        else:
            n.ptr = abase + n.buf[0]
            n.bstride = (1 << n.rank) if n.batched else 0

    def recp(n):
        return rbase + n.rec * 16 if scaled else 0

    blob = bytearray()

    def put(structs):
        nonlocal blob
        start = (len(blob) + ALIGN - 1) // ALIGN * ALIGN
        blob += b"\0" * (start - len(blob))
        for st in structs:
            blob += bytes(st)
        return start

    prog.build = []
    if image.builds:
        bdescs, block0 = [], 0
        for t, v0, v1 in image.builds:
            bd = tables[t].spec.desc(tbase + image.off[t] * esize, v0, v1)
            bd.block0 = block0
            block0 += bd.nblocks
            bdescs.append(bd)
        prog.build.append((Launch(op=_lib.TO_OP_LEAF_BUILD, count=len(bdescs), grid=block0), put(bdescs)))

    def group_launches(group, phase):
        """The joins of one group as one launch per kernel variant; permutes before products,
        split sums before their finishing."""
        keyed = {}
        for i in group:
            n = nodes[i]
            for kind, op, variant, lds, st, nblk in join_records(n, nodes, W, esize, scaled, abase,
                                                                 scratch.get(i, {}), recp, one_at):
                if kind == "permute":
                    work = (2 * esize * (int(st.nbatch) << int(st.rank)), 0)
                elif kind in ("fold", "gemm"):
                    work = join_traffic(n, nodes, W, esize)
                elif kind == "pair":
                    work = (sum((1 << nodes[c].rank) * (W if nodes[c].batched else 1) for c in _reads(n)) * esize,
                            sum(join_traffic(nodes[c], nodes, W, esize)[1]
                                for c in [i] + [f.idx for *_, f in n.geom["var"]["sides"] if f is not None]))
                else:
                    work = (0, 0)
                keyed.setdefault((schedule.KIND_ORDER[kind], op, variant), []).append((kind, st, nblk, lds, i, work))
        for key in sorted(keyed):
            grp = sorted(keyed[key], key=lambda r: -block_cost(r[1]))
            block0, lds, wb, wf = 0, 0, 0, 0
            for kind, st, nblk, l, i, work in grp:
                st.block0 = block0
                block0 += nblk
                lds = max(lds, l)
                wb += work[0]
                wf += work[1]
            off = put([r[1] for r in grp])
            phase.append((grp[0][0], Launch(op=key[1], variant=key[2], count=len(grp), grid=block0, lds=lds), off,
                          grp[0][4] if len(grp) == 1 else None, (wb, wf)))

    def put_raw(data):
        nonlocal blob
        start = (len(blob) + ALIGN - 1) // ALIGN * ALIGN
        blob += b"\0" * (start - len(blob)) + data
        return start

    def run_phase(batched, phase):
        for programs_, joins in phase_groups(nodes, batched, order, programs):
            if programs_:
                tree_launch(programs_, phase, batched)
            if joins:
                group_launches(joins, phase)

    def tree_launch(mine, phase, batched):
        """One launch of programs, the longest streams first."""
        block0, wb, wf, built, descs = 0, 0, 0, [], []
        waves = TREE_WAVES_MANY if batched and W >= TREE_MANY else TREE_WAVES
        for p in mine:
            built.append(tree_words(p, nodes, waves, lambda n: n.rec if scaled else 0,
                                    (one_at[0], one_rec if scaled else 0)) + (p,))
            for i in p.members:
                b, f = join_traffic(nodes[i], nodes, W, esize)
                wb, wf = wb + b, wf + f
        for words, streams, p in sorted(built, key=lambda b: -b[1].shape[1]):
            td = _lib.TreeDesc(ntask=streams.shape[1], nslots=len(p.slot) if scaled else 0, block0=block0,
                               nblocks=W if batched else 1)
            block0 += td.nblocks
            descs.append((td, put_raw(words.tobytes()), put_raw(streams.tobytes())))
        at = put_raw(bytes(ctypes.sizeof(_lib.TreeDesc) * len(descs)))
        tree_places.append((at, descs))
        phase.append(("tree", Launch(op=_lib.TO_OP_FOLD_TREE, count=len(descs), grid=block0, iaux0=waves,
                                     lds=max(16, max(p.lds for p in mine))), at, None, (wb, wf)))

    tree_places = []

    prog.self_start = True

    def clear(a, b):
        return ("clear", Launch(op=_lib.TO_OP_SCALE_CLEAR, grid=max(1, min(1024, -(-(b - a) // 256))),
                                aux0=rbase + a * 16, iaux0=b - a), None, None, (0, 0))

    pro, wave = [], []
    if scaled and prog.rec_ranges[1] > prog.rec_ranges[0]:
        pro.append(clear(*prog.rec_ranges[:2]))
    run_phase(False, pro)
    root = nodes[-1]
    prog.root_const = not root.batched
    leaf_descs, block0 = [], 0
    for n in nodes:
        if n.is_leaf and n.batched:
            ld = LeafDesc(src=tbase + image.off[n.tensor] * esize, dst=n.ptr,
                          coef=prog.coef.data_ptr() + image.coef_off[n.tensor] * 8, rec=recp(n),
                          exp0=image.exp0.get(n.tensor, 0), rank=n.rank, ngroups=num_groups, nbatch=W, block0=block0,
                          nblocks=int(min(1024, -(-(W << n.rank) // 256))))
            block0 += ld.nblocks
            leaf_descs.append(ld)
    nclear = nrec - clear_rec0 if scaled else 0
    if leaf_descs or nclear:
        clear_blocks = min(1024, -(-nclear // 256))
        wave.append(("leaf", Launch(op=_lib.TO_OP_WAVE_BEGIN, count=len(leaf_descs), grid=block0 + clear_blocks,
                                    aux0=rbase + clear_rec0 * 16 if nclear else 0, iaux0=nclear, iaux1=block0,
                                    aux3=wave_params),
                     put(leaf_descs), None, (sum(esize * (W << ld.rank) for ld in leaf_descs), 0)))
    run_phase(True, wave)
    root_launch = Launch(op=_lib.TO_OP_ROOT_REDUCE, variant=1, grid=1, aux0=root.ptr, aux1=recp(root),
                         iaux1=prog.host_accum.data_ptr() if prog.host_accum is not None else 0,
                         aux2=prog.accum.data_ptr(), aux3=wave_params + (16 if prog.root_const else 0),
                         iaux0=1 if prog.root_const else W)
    (pro if prog.root_const else wave).append(("root", root_launch, None, None, (0, 0)))

    prog.blob = device_alloc(max(1, len(blob)))
    bbase = prog.blob.data_ptr()
    for at, descs in tree_places:
        for td, ops_at, tasks_at in descs:
            td.ops, td.tasks, td.recs = bbase + ops_at, bbase + tasks_at, rbase
        raw = b"".join(bytes(td) for td, _, _ in descs)
        blob[at:at + len(raw)] = raw
    prog.blob_host = np.frombuffer(bytes(blob) or b"\0", dtype=np.uint8).copy()
    for L, off in prog.build:
        L.descs = bbase + off
    prog.build = [L for L, _ in prog.build]
    prog.prologue_info, prog.wave_info, prog.prologue_work, prog.wave_work = [], [], [], []
    for lst, out, info, work in ((pro, prog.prologue, prog.prologue_info, prog.prologue_work),
                                 (wave, prog.wave, prog.wave_info, prog.wave_work)):
        for kind, L, off, nidx, w in lst:
            if off is not None:
                L.descs = bbase + off
            out.append(L)
            info.append((kind, nidx))
            work.append(w)
    joins = [n for n in nodes if not n.is_leaf]
    prog.stats = dict(
        nodes=len(nodes), joins=len(joins), batched_joins=sum(1 for n in joins if n.batched),
        splitk=sum(1 for n in joins if n.geom["var"].get("lsplit")),
        gemm=sum(1 for n in joins if n.geom["var"]["kind"] == "gemm"),
        tree_joins=sum(len(p.members) for p in programs),
        arena_bytes=peak, table_bytes=int(image.host.nbytes),
        # leaves described for the device (a vector of ones among them needs no table)
        device_built_leaves=sum(1 for t in tables.values() if t.spec is not None),
        launches_prologue=len(prog.prologue), launches_wave=len(prog.wave))
    return prog


# many-instance batches: programs keep to this much LDS, so that two blocks of 16 waves share
# a CU
TREE_LDS_BATCH = 64 * 1024


def analyse_batch(instances, esize, regroup=True):
    """Per (tree, tables) of unsliced plans: its folded nodes with their forms, programs,
    memory plan and arena region; None when a plan cannot be folded."""
    per = []
    for tree, tables in instances:
        folded = analyse(tree, tables, esize, regroup) if has_copies(tables) else None
        if folded is None:
            return None
        nodes, missing = folded
        if any(n.batched for n in nodes):
            raise ValueError("batched instances must be unsliced plans")
        try:
            choose_all(nodes, 1, esize, launch_bound=True)
        except TooWide:
            return None
        programs = tree_programs(nodes, 1, esize, esize == 4, TREE_LDS_BATCH)
        peak, scratch = plan_memory(nodes, 1, esize, "level", programs)
        words = sum(len(p.members) for p in programs) * 4 * _lib.TO_TREE_WORDS
        per.append(dict(nodes=nodes, missing=missing, tables=tables, programs=programs, scratch=scratch,
                        region=(max(peak, ALIGN) + ALIGN - 1) // ALIGN * ALIGN,
                        fixed=sum(t.size for t in tables.values()) * esize + 1024 * len(nodes) + words))
    return per


def compile_batch(per, entry_type, device_alloc, arena, host_alloc):
    """One grouped schedule (``batch.BatchProgram``) of analysed instances: step k runs the
    k-th group of every instance -- its programs in one launch, its other joins in one launch
    per kernel form -- through the given arena, every instance in its own region; an
    instance's root goes to its accumulator right after its last step.  The accumulators and
    the start time lie in host memory that the device writes (``host_alloc``)."""
    from .batch import MAP_MIN_DESCS, BatchProgram

    esize = 8 if entry_type == _lib.TO_F64 else 4
    scaled = entry_type == _lib.TO_F32S
    fdtype = np.float64 if esize == 8 else np.float32
    prog = BatchProgram()
    prog.count, prog.per, prog.arena = len(per), per, arena
    # leaf tables of all instances in one buffer, a stored 1.0 last
    chunks, top, bases = [], 0, []
    prog.leaf_factors = []
    for inst in per:
        inst["image"] = im = schedule.leaf_image(inst["nodes"], inst["tables"], 0, scaled, fdtype)
        bases.append(top)
        chunks.append(im.host)
        top += im.host.size
        prog.leaf_factors.append((im.factor[0], im.factor[1] + inst["missing"]))
    chunks.append(np.ones(1, fdtype))
    prog.table_host = np.concatenate(chunks)
    one = top
    # scale records: constant leaves and the 1.0, then what the launches write
    nrec, prog.rec_init = 1, [(0, 0)]
    for inst in per:
        for n in inst["nodes"]:
            if n.is_leaf:
                n.rec, n.rec_stride = nrec, 0
                if scaled:
                    prog.rec_init.append((nrec, inst["image"].exp0[n.tensor]))
                nrec += 1
    join_rec0 = nrec
    for inst in per:
        inst["in_lds"] = {i for p in inst["programs"] for i in p.members if i != p.root}
        for n in inst["nodes"]:
            if not n.is_leaf and n.idx not in inst["in_lds"]:
                n.rec, n.rec_stride = nrec, 0
                nrec += 1
    prog.rec_count = nrec if scaled else 0
    prog.table = device_alloc(prog.table_host.nbytes)
    prog.recs = device_alloc(max(1, nrec) * 16)
    prog.accum = host_alloc(len(per) * ctypes.sizeof(_lib.Accum))
    prog.start = host_alloc(64)
    tbase, rbase, abase = prog.table.data_ptr(), prog.recs.data_ptr(), arena.data_ptr()
    one_at = (tbase + one * esize, rbase if scaled else 0)

    def recp(n):
        return rbase + n.rec * 16 if scaled else 0

    blob = bytearray()

    def put(data):
        nonlocal blob
        start = (len(blob) + ALIGN - 1) // ALIGN * ALIGN
        blob += b"\0" * (start - len(blob)) + data
        return start

    base, builds, steps, roots = 0, [], [], {}
    for k, inst in enumerate(per):
        nodes = inst["nodes"]
        at, im = bases[k], inst["image"]
        for n in nodes:
            n.bstride = 0
            if n.is_leaf:
                n.ptr = tbase + (at + im.off[n.tensor]) * esize
            elif n.idx not in inst["in_lds"]:
                n.ptr = abase + base + n.buf[0]
        for t, v0, v1 in im.builds:
            bd = inst["tables"][t].spec.desc(tbase + (at + im.off[t]) * esize, v0, v1)
            bd.block0 = builds[-1].block0 + builds[-1].nblocks if builds else 0
            builds.append(bd)
        groups = phase_groups(nodes, False, "level", inst["programs"])
        for i, grp in enumerate(groups):
            while len(steps) <= i:
                steps.append(([], {}))
            for p in grp[0]:
                steps[i][0].append((p, nodes))
            for j in grp[1]:
                scratch = {key: (base + blk[0], blk[1]) for key, blk in inst["scratch"].get(j, {}).items()}
                for kind, op, variant, lds, st, nblk in join_records(nodes[j], nodes, 1, esize, scaled, abase, scratch,
                                                                     recp, one_at, True):
                    work = join_traffic(nodes[j], nodes, 1, esize) if kind in ("fold", "gemm") else (0, 0)
                    if kind == "permute":
                        work = (2 * esize << int(st.rank), 0)
                    steps[i][1].setdefault((schedule.KIND_ORDER[kind], op, variant), []).append((kind, st, nblk, lds, work))
        root = nodes[-1]
        rd = _lib.RootDesc(root=root.ptr, rec=recp(root), acc=prog.accum.data_ptr() + k * ctypes.sizeof(_lib.Accum))
        roots.setdefault(len(groups) - 1, []).append(rd)
        base += inst["region"]

    build_at = put(b"".join(bytes(b) for b in builds)) if builds else None
    pending = [(Launch(op=_lib.TO_OP_BATCH_BEGIN, grid=max(1, min(64, -(-len(per) // 256))), aux2=prog.accum.data_ptr(),
                       aux3=prog.start.data_ptr(), iaux0=len(per)), None, None, ("begin", -1), (0, 0))]
    if scaled and nrec > join_rec0:
        pending.append((Launch(op=_lib.TO_OP_SCALE_CLEAR, grid=max(1, min(1024, -(-(nrec - join_rec0) // 256))),
                               aux0=rbase + join_rec0 * 16, iaux0=nrec - join_rec0), None, None, ("clear", -1), (0, 0)))
    tree_places = []

    def bmap(blocks):
        return put(np.repeat(np.arange(len(blocks), dtype=np.int32), blocks).tobytes()) \
            if len(blocks) >= MAP_MIN_DESCS else None

    for i, (trees, keyed) in enumerate(steps):
        if trees:
            waves = TREE_WAVES_MANY if len(trees) >= TREE_MANY else TREE_WAVES
            built, wb, wf = [], 0, 0
            for p, nodes in trees:
                built.append(tree_words(p, nodes, waves, lambda n: n.rec if scaled else 0, (one_at[0], 0)) + (p,))
                for j in p.members:
                    b, f = join_traffic(nodes[j], nodes, 1, esize)
                    wb, wf = wb + b, wf + f
            built.sort(key=lambda b: -b[1].shape[1])  # the longest streams start first
            descs = []
            for j, (words, streams, p) in enumerate(built):
                td = _lib.TreeDesc(ntask=streams.shape[1], nslots=len(p.slot) if scaled else 0, block0=j, nblocks=1)
                descs.append((td, put(words.tobytes()), put(streams.tobytes())))
            at = put(bytes(ctypes.sizeof(_lib.TreeDesc) * len(descs)))
            tree_places.append((at, descs))
            pending.append((Launch(op=_lib.TO_OP_FOLD_TREE, count=len(descs), grid=len(descs), iaux0=waves,
                                   lds=max(16, max(b[2].lds for b in built))), at, bmap([1] * len(descs)), ("tree", i),
                            (wb, wf)))
        for key in sorted(keyed):
            grp = sorted(keyed[key], key=lambda r: -block_cost(r[1]))
            block0 = 0
            for _, st, nblk, _, _ in grp:
                st.block0 = block0
                block0 += nblk
            at = put(b"".join(bytes(r[1]) for r in grp))
            pending.append((Launch(op=key[1], variant=key[2], count=len(grp), grid=block0, lds=max(r[3] for r in grp)),
                            at, bmap([r[2] for r in grp]), (grp[0][0], i),
                            (sum(r[4][0] for r in grp), sum(r[4][1] for r in grp))))
        if i in roots:
            at = put(b"".join(bytes(r) for r in roots[i]))
            pending.append((Launch(op=_lib.TO_OP_ROOT_STORE, count=len(roots[i]), grid=max(1, -(-len(roots[i]) // 256))),
                            at, None, ("root", i), (0, 0)))
    prog.blob = device_alloc(max(1, len(blob)))
    bbase = prog.blob.data_ptr()
    for at, descs in tree_places:
        for td, ops_at, tasks_at in descs:
            td.ops, td.tasks, td.recs = bbase + ops_at, bbase + tasks_at, rbase
        raw = b"".join(bytes(td) for td, _, _ in descs)
        blob[at:at + len(raw)] = raw
    prog.blob_host = np.frombuffer(bytes(blob) or b"\0", dtype=np.uint8).copy()
    prog.build = [] if build_at is None else [
        Launch(op=_lib.TO_OP_LEAF_BUILD, count=len(builds), grid=builds[-1].block0 + builds[-1].nblocks,
               descs=bbase + build_at)]
    prog.work = []
    for L, at, mat, info, work in pending:
        if at is not None:
            L.descs = bbase + at
        if mat is not None:
            L.aux1 = bbase + mat
        prog.launches.append(L)
        prog.info.append(info)
        prog.work.append(work)
    kinds = {}
    for kind, _ in prog.info:
        kinds[kind] = kinds.get(kind, 0) + 1
    prog.stats = dict(instances=len(per), steps=len(steps), launches=len(prog.launches),
                      joins=sum(1 for inst in per for n in inst["nodes"] if not n.is_leaf),
                      arena_bytes=base, launches_per_kind=kinds)
    return prog
