"""The MI355X ``tensor_library``: a drop-in ``BaseTensorAPI`` backed by HIP kernels.

Mirrors the plugin interface the reference's ``execution.run`` drives
(``tensor_network/tensor_apis/base_api.py:8-28``; registry ``tensor_network/__init__.py:12-16``):

* ``add_argument(key, value)``: ``entry_type`` (``float64`` = plain FP64 executor,
  ``float32`` = FP32 with per-tensor power-of-two scaling), ``thread_limit`` (accepted;
  host threads do no arithmetic here), ``max_batch``, ``mem_limit`` (bytes of device
  memory the executor may use), ``graph`` (capture waves in a HIP graph), ``regroup``,
  ``autotune`` (time the launch shapes of new product/permute shapes before compiling);
  any other key raises ``ValueError`` (``base_api.py:9-12``).
* ``contract_sliced(plan, num_slice_limit)``: all slices of the plan, batched in waves on
  the device, summed in FP64 (mantissa, exponent) -- the override pattern of
  ``jax_apis.py:316-322``; returns a Python float.
* ``contract(network, tree)``: one (possibly sliced) network; returns a 0-d array.
* ``create_tensor`` / ``reshape`` / ``transpose`` build leaf values on the host (leaves
  are tiny), ``tensordot`` contracts two tensors on the device (the per-join primitive
  ``network.identify`` calls, ``tensor_network.pyx:152-154``).

Device memory is allocated through PyTorch; the arithmetic runs only in the HIP library.
If the library or the GPU is missing, construction raises.
"""

import contextlib
import ctypes
import math
import threading

import numpy as np

from . import _lib, fold, schedule
from .api import BaseTensorAPI, OutOfMemoryError
from .tree import TreeContext


class DeviceTensor:
    """A dense tensor in device memory (entry type of its API), optionally with a
    power-of-two scale record (FP32 mode)."""

    def __init__(self, data, shape, rec=None, api=None):
        self.data = data
        self.shape = tuple(shape)
        self.rec = rec
        self._api = api

    @property
    def rank(self):
        return len(self.shape)

    def numpy(self):
        vals = self.data.double().cpu().numpy().reshape(self.shape)
        if self.rec is not None:
            exp = int(self.rec.cpu().numpy().view(np.int64)[0])
            vals = np.ldexp(vals, exp)
        return vals

    def __getitem__(self, item):
        return self.numpy()[item]


class Result:
    """A count as FP64 mantissa and int64 exponent (value = mant * 2^exp)."""

    def __init__(self, mant, exp, slices):
        self.mant, self.exp, self.slices = float(mant), int(exp), int(slices)

    @property
    def value(self):
        try:
            return math.ldexp(self.mant, self.exp)
        except OverflowError:
            return math.copysign(math.inf, self.mant)

    @property
    def log10(self):
        if self.mant == 0:
            return -math.inf
        return math.log10(abs(self.mant)) + self.exp * math.log10(2.0)


class Executable:
    """A compiled plan resident on the device.  ``run()`` is one full contraction: reset
    the accumulator, prologue (slice-invariant subtrees), then every wave of slices,
    replayed from HIP graphs when the API's ``graph`` option is on."""

    # a run of at most this many launches is one graph: between graphs the device waits for
    # the host
    ONE_GRAPH_LAUNCHES = 512

    def __init__(self, api, prog, total_slices, once=False):
        self.api = api
        self.prog = prog
        self.total = total_slices
        self.nwaves = 0 if prog.root_const else -(-total_slices // prog.nbatch)
        begin = _lib.Launch(op=_lib.TO_OP_STEP_BEGIN, grid=1, aux2=prog.accum.data_ptr(),
                            aux3=prog.params.data_ptr())
        self._step, self._wave = [begin] + list(prog.prologue), list(prog.wave)
        self._graphs = []
        # what a run replays, in order: graphs, or launch lists run one by one
        first = list(prog.prologue) if prog.self_start else self._step
        runs = [first] + [self._wave] * self.nwaves
        if sum(len(r) for r in runs) <= self.ONE_GRAPH_LAUNCHES:
            runs = [sum(runs, [])]
        # a plan that runs once only pays for capturing waves that repeat
        captured = {}
        self._runs = []
        # the sum in host memory, and its word (None: the sum stays on the device, and a run's
        # first launch resets what it needs)
        self._sum = self._sum_word = None
        if prog.host_accum is not None:
            self._sum = _lib.Accum.from_address(prog.host_accum.data_ptr())
            self._sum_word = ctypes.c_void_p(prog.host_accum.data_ptr() + _lib.Accum.pad.offset)
        self._stream = ctypes.c_void_p(api._stream.cuda_stream)
        # runs queued since the last wait, and the value of the sum's word that ends them
        self._queued, self._word = 0, 0
        # whether the device's wave counter stands at the first slice once what is queued is
        # done: a run leaves it there, one cut short does not
        self._whole = True
        self._lent = False  # whether a caller has the launches, and may run them by itself
        # whether the uploads that made the plan resident may still be under way
        self._fresh = True
        self._sums = sum(L.op == _lib.TO_OP_ROOT_REDUCE for r in runs for L in r)
        for r in runs:
            if id(r) not in captured:
                use = api._use_graph and r and (not once or (r is self._wave and self.nwaves > 2))
                captured[id(r)] = (self._capture(r) if use else None, r)
            self._runs.append(captured[id(r)])

    def _capture(self, launches):
        arr = _lib.launch_array(launches)
        graph = ctypes.c_void_p()
        _lib.check(self.api._lib.to_graph_create(ctypes.addressof(arr), len(launches), self.api._entry_type,
                                                 ctypes.c_void_p(self.api._stream.cuda_stream),
                                                 ctypes.byref(graph)), "to_graph_create")
        self._graphs.append(graph)
        return graph

    def _launch_graph(self, graph):
        _lib.check(self.api._lib.to_graph_launch(graph, self._stream), "to_graph_launch")

    @property
    def step_launches(self):
        """The launches that open a run: its start, then the prologue."""
        self._lent = True
        return self._step

    @property
    def wave_launches(self):
        """The launches of one wave of slices."""
        self._lent = True
        return self._wave

    def enqueue(self):
        """Queue one full contraction on the API's stream (no synchronisation)."""
        if self._sum is not None:
            if not self._whole:
                # an earlier run was cut short (a failed launch, an interrupt): nothing of it is
                # counted, and the device's counter may stand between its waves
                self.api.synchronize()
                self._queued = 0
            if self._lent or not self._whole:
                self.api._upload(self.prog.params, self.counters(self.total))
            if not self._queued:
                self._word = self._sum.pad
        self._whole = False
        for graph, launches in self._runs:
            if graph is not None:
                self._launch_graph(graph)
            else:
                self.api._run(launches)
        if self._sum is not None:
            self._queued += 1
            self._word += self._sums
        self._whole = True

    @staticmethod
    def counters(total):
        """The device's counters: the wave's first slice and the number of slices, and the same
        of the prologue."""
        return np.array([0, total, 0, 1], dtype=np.int64).tobytes()

    def result(self):
        """Synchronise and read the (mantissa, exponent) slice sum."""
        api = self.api
        acc = self._sum
        if acc is not None:
            if not self._whole:
                raise RuntimeError("the last run was cut short while it was queued")
            if self._lent or not self._sums:  # (launches that a caller runs count in the word too)
                api.synchronize()
            elif self._queued:
                _lib.check(api._lib.to_wait(self._sum_word, self._word, self._stream), "to_wait")
                if acc.pad < self._word:
                    raise RuntimeError("the device is idle and has not written the sum")
            if self._queued or self._lent:
                self._queued, self._fresh = 0, False
        else:
            api.synchronize()
            self._fresh = False
            with api._torch.cuda.stream(api._stream):
                acc_bytes = self.prog.accum[: ctypes.sizeof(_lib.Accum)].cpu().numpy().tobytes()
            acc = _lib.Accum.from_buffer_copy(acc_bytes)
        fm, fe = getattr(self.prog, "leaf_factor", (1.0, 0))
        res = Result(acc.mant * fm, acc.exp + fe, acc.count)
        api.last_result = res
        api.last_stats = dict(self.prog.stats, nbatch=self.prog.nbatch, waves=self.nwaves, slices=self.total)
        return res

    def run(self):
        self.enqueue()
        return self.result()

    def _in_flight(self):
        """Whether the device may still write this object's memory."""
        return bool(getattr(self, "_queued", 0) or getattr(self, "_fresh", False) or not getattr(self, "_whole", True))

    def close(self):
        if self._graphs or self._in_flight():
            self.api.synchronize()  # the sum's word is written by a kernel that has yet to end
            self._queued, self._fresh = 0, False
        for g in self._graphs:
            self.api._lib.to_graph_destroy(g)
        self._graphs = []
        self._runs = [(None, launches) for _, launches in self._runs]

    def __del__(self):
        # runs, or uploads, that nobody waited for write to this object's memory until they end
        if self._in_flight():
            self.api.synchronize()


class BatchExecutable:
    """A batch of unsliced plans resident on the device, admitted in waves sized to the
    device budget: one grouped schedule (one HIP graph) per wave, the waves run in order
    through one shared arena.  ``run()`` contracts all of them and returns their Results and
    per-instance completion times (s from the batch start, device clock)."""

    def __init__(self, api, progs, arena=None):
        self.api = api
        self.progs = list(progs)
        self.prog = self.progs[0]
        self.arena = arena
        self.count = sum(p.count for p in self.progs)
        self._graphs = []
        self._queued = True  # (the uploads that made the plans resident)
        if api._use_graph:
            for prog in self.progs:
                arr = _lib.launch_array(prog.launches)
                graph = ctypes.c_void_p()
                _lib.check(api._lib.to_graph_create(ctypes.addressof(arr), len(prog.launches), api._entry_type,
                                                    ctypes.c_void_p(api._stream.cuda_stream), ctypes.byref(graph)),
                           "to_graph_create")
                self._graphs.append(graph)
        khz = ctypes.c_int(0)
        _lib.check(api._lib.to_wall_clock_khz(ctypes.byref(khz)), "to_wall_clock_khz")
        self.clock_hz = khz.value * 1e3

    @property
    def launches(self):
        return [L for prog in self.progs for L in prog.launches]

    @property
    def work(self):
        return [w for prog in self.progs for w in prog.work]

    def enqueue(self):
        self._queued = True
        if self._graphs:
            for graph in self._graphs:
                _lib.check(self.api._lib.to_graph_launch(graph, ctypes.c_void_p(self.api._stream.cuda_stream)),
                           "to_graph_launch")
        else:
            for prog in self.progs:
                self.api._run(prog.launches)

    def results(self):
        api = self.api
        api.synchronize()
        self._queued = False
        size = ctypes.sizeof(_lib.Accum)
        res, ends = [], []
        # (no copies where the accumulators lie in host memory)
        with api._torch.cuda.stream(api._stream):
            start = int(self.progs[0].start[:8].cpu().numpy().view(np.int64)[0])
            for prog in self.progs:
                raw = prog.accum[: prog.count * size].cpu().numpy().tobytes()
                accs = [_lib.Accum.from_buffer_copy(raw[i * size:(i + 1) * size]) for i in range(prog.count)]
                res += [Result(a.mant * fm, a.exp + fe, a.count) for a, (fm, fe) in zip(accs, prog.leaf_factors)]
                ends += [a.pad for a in accs]
        lat = [(e - start) / self.clock_hz for e in ends]
        return res, lat

    def run(self):
        self.enqueue()
        return self.results()

    def close(self):
        if self._queued:
            self.api.synchronize()
            self._queued = False
        for graph in self._graphs:
            self.api._lib.to_graph_destroy(graph)
        self._graphs = []

    def __del__(self):
        # (see Executable)
        if getattr(self, "_queued", False):
            self.api.synchronize()


def copy_weights(tensor):
    """(w(not x), w(x), whether it has axes) of a COPY tensor, else None."""
    from .network import VariableTensor

    return tensor.weights + (tensor.rank > 0,) if isinstance(tensor, VariableTensor) else None


def leaf_spec_table(tensor, lookup, ngroups):
    """The LeafTable of an OR or variable leaf whose table the device writes, with its axes
    reordered and its row lookup exactly as ``SliceSequence.reordered_tensor`` gives them
    (``tensor.py:95-119``); None for other leaves."""
    from .network import OrTensor, VariableTensor

    copy = None
    if isinstance(tensor, VariableTensor):
        w_neg, w_pos = tensor.weights
        copy = (w_neg, w_pos, tensor.rank > 0)
        kind, kw = _lib.TO_LEAF_VAR, dict(w_neg=w_neg, w_pos=w_pos)
    elif isinstance(tensor, OrTensor):
        kind, kw = _lib.TO_LEAF_OR, dict(positive=tensor.literals_positive, output_index=tensor.output_index)
    else:
        return None
    rank = tensor.rank
    sliced = [i for i in range(rank) if i in lookup]
    unsliced = [i for i in range(rank) if i not in lookup]
    coef = [0] * ngroups
    offset = 1
    for i in reversed(sliced):
        coef[lookup[i]] += offset
        offset *= 2
    spec = schedule.LeafSpec(kind, rank, sliced + unsliced, **kw)
    return schedule.LeafTable(None, coef, len(unsliced), spec, copy=copy)


class HipAPI(BaseTensorAPI):
    def __init__(self, device=0):
        import torch

        self._torch = torch
        self._lib = _lib.load()
        if not torch.cuda.is_available():
            raise RuntimeError("HipAPI needs a ROCm GPU; none is visible")
        self._device = torch.device("cuda", device)
        self._stream = torch.cuda.Stream(device=self._device)
        self._entry_type = _lib.TO_F64
        self._thread_limit = None
        self._max_batch = 1 << 16
        self._mem_limit = None
        self._use_graph = True
        self._regroup = True
        self._autotune = False
        self._signal_lock = threading.Lock()
        self._signals = 0
        self._signal_word = torch.zeros(1, dtype=torch.int64, pin_memory=True)  # see ``finish``
        self._device_leaves = True
        # launch shapes tuned on this GPU model (autotune.py), used where a shape is known
        from . import autotune

        schedule.TUNED.update(autotune.load())
        self.last_result = None
        self.last_stats = {}

    # -- plugin interface ---------------------------------------------------------

    def add_argument(self, key, value):
        if key == "entry_type":
            types = {"float64": _lib.TO_F64, "float32": _lib.TO_F32S}
            if value not in types:
                raise ValueError("Unknown hip type %s" % value)
            self._entry_type = types[value]
        elif key == "thread_limit":
            self._thread_limit = value
        elif key == "max_batch":
            self._max_batch = max(1, int(value))
        elif key == "mem_limit":
            self._mem_limit = None if value is None else int(value)
        elif key == "graph":
            self._use_graph = bool(value)
        elif key == "regroup":
            self._regroup = bool(value)
        elif key == "autotune":
            self._autotune = bool(value)
        elif key == "device_leaves":
            self._device_leaves = bool(value)
        else:
            super().add_argument(key, value)

    def get_entry_size(self):
        return 8 if self._entry_type == _lib.TO_F64 else 4

    def warm(self):
        a = self.create_tensor((2,), 2)
        self.tensordot(a, a, ([0], [0]))
        self.synchronize()

    def create_tensor(self, shape, default_value=None):
        if default_value is None:
            return np.empty(shape, dtype=np.float64)
        return np.full(shape, default_value, dtype=np.float64)

    def reshape(self, tensor, new_shape):
        return np.reshape(tensor, new_shape)

    def transpose(self, tensor, perm):
        return np.transpose(tensor, axes=perm)

    # -- device helpers -----------------------------------------------------------

    @property
    def _esize(self):
        return self.get_entry_size()

    def _alloc(self, nbytes):
        try:
            return self._torch.empty(max(1, int(nbytes)), dtype=self._torch.uint8, device=self._device)
        except self._torch.OutOfMemoryError:
            raise OutOfMemoryError

    def _alloc_host(self, nbytes):
        """Host memory that the device writes (pinned)."""
        return self._torch.empty(max(1, int(nbytes)), dtype=self._torch.uint8, pin_memory=True)

    # larger data go through a copy engine
    UPLOAD_BYTES = 12 * 1024

    @contextlib.contextmanager
    def _settled(self):
        """Queued work is waited for before an exception drops the memory it uses."""
        try:
            yield
        except BaseException:
            self.synchronize()
            raise

    def _upload(self, dst, host_bytes):
        """Copy to the device in stream order: small data are still on their way on return."""
        n = len(host_bytes)
        if n <= self.UPLOAD_BYTES and n % 4 == 0:
            _lib.check(self._lib.to_upload(ctypes.c_void_p(dst.data_ptr()), ctypes.c_char_p(bytes(host_bytes)), n,
                                           ctypes.c_void_p(self._stream.cuda_stream)), "to_upload")
            return
        src = self._torch.from_numpy(np.frombuffer(host_bytes, dtype=np.uint8).copy())
        with self._torch.cuda.stream(self._stream):
            dst[: src.numel()].copy_(src, non_blocking=False)

    def _run(self, launches):
        if not launches:
            return
        arr = _lib.launch_array(launches)
        rc = self._lib.to_run(ctypes.addressof(arr), len(launches), self._entry_type,
                              ctypes.c_void_p(self._stream.cuda_stream))
        if rc == _lib.TO_ERR_OOM:
            raise OutOfMemoryError
        _lib.check(rc, "to_run")

    def synchronize(self):
        _lib.check(self._lib.to_synchronize(ctypes.c_void_p(self._stream.cuda_stream)), "to_synchronize")

    def finish(self):
        """Wait until the work queued so far is done, by a word the device writes at its end."""
        with self._signal_lock:  # the words' order is the stream's
            self._signals += 1
            value = self._signals
            word = ctypes.c_void_p(self._signal_word.data_ptr())
            stream = ctypes.c_void_p(self._stream.cuda_stream)
            _lib.check(self._lib.to_signal(word, value, stream), "to_signal")
        _lib.check(self._lib.to_wait(word, value, stream), "to_wait")

    def _budget(self):
        # free device memory plus what torch's caching allocator holds without using it
        free, _total = self._torch.cuda.mem_get_info(self._device)
        cached = self._torch.cuda.memory_reserved(self._device) - self._torch.cuda.memory_allocated(self._device)
        budget = int((free + max(0, cached)) * 0.85)
        if self._mem_limit is not None:
            budget = min(budget, self._mem_limit)
        return budget

    # -- compiled execution ---------------------------------------------------------

    def choose_folded_batch(self, folded, tree, tables, total_slices):
        """Largest slice batch W of a folded plan whose arena fits the device budget (0: it
        runs edge by edge).  A plan is refused where its tensors, one axis per edge, would not
        fit one slice at a time: whether a caller has to slice more does not depend on how the
        plan is executed."""
        budget = self._budget()
        nodes, _ = folded
        fixed = sum(t.size for t in tables.values()) * self._esize
        if fixed + schedule.peak_bound(tree, self._esize) > budget:
            self.choose_batch(schedule.analyse(tree, tables, self._regroup), tables, 1)
        W = max(1, min(self._max_batch, total_slices))
        try:
            while W and fold.peak_bytes(nodes, W, self._esize) + fixed > budget:
                W //= 2
        except fold.TooWide:
            return 0
        return W

    def choose_batch(self, nodes, tables, total_slices):
        """Largest slice batch W (<= max_batch) whose arena fits the device budget; raises
        OutOfMemoryError when even one slice does not fit."""
        budget = self._budget()
        fixed = sum(t.size for t in tables.values()) * self._esize
        W = max(1, min(self._max_batch, total_slices))
        while True:
            peak = schedule.peak_bytes(nodes, tables, W, self._entry_type)
            if peak + fixed <= budget:
                return W
            if W == 1:
                raise OutOfMemoryError
            W = max(1, W // 2)

    def _compile(self, tree, tables, num_groups, total_slices, group_levels=True, once=False):
        """Compile and upload a plan; returns an ``Executable``.  ``group_levels=False``
        keeps one launch per join (per-join timing); ``once``: the plan runs a single time."""
        folded = fold.analyse(tree, tables, self._esize, self._regroup) if fold.has_copies(tables) else None
        W = self.choose_folded_batch(folded, tree, tables, total_slices) if folded is not None else 0
        if W:
            if self._tune(folded[0], W):
                folded[0][-1].layout = None  # (laid out with the shapes known before)
            prog = fold.compile_program(folded, tables, num_groups, self._entry_type, W, self._alloc, group_levels,
                                        self._alloc_host)
            return self._resident(prog, total_slices, once)
        nodes = schedule.analyse(tree, tables, self._regroup)
        W = self.choose_batch(nodes, tables, total_slices)
        self._tune(nodes, W)
        prog = schedule.compile_program(tree, tables, num_groups, self._entry_type, W, self._alloc,
                                        regroup=self._regroup, group_levels=group_levels)
        return self._resident(prog, total_slices, once)

    def _tune(self, nodes, W):
        """Time the launch shapes that a plan is the first to need (``autotune`` option); returns
        how many."""
        if not self._autotune:
            return 0
        from . import autotune

        with self._settled():
            tuned = autotune.tune_plan(self, nodes, W, schedule.TUNED)
        if tuned:
            autotune.save(schedule.TUNED)
        return tuned

    def _resident(self, prog, total_slices, once):
        """Upload a compiled plan; returns its ``Executable``."""
        with self._settled():
            self._upload(prog.table, prog.table_host.tobytes())
            self._upload(prog.coef, prog.coef_host.tobytes())
            self._upload(prog.blob, prog.blob_host.tobytes())
            self._run(prog.build)  # OR / variable leaf tables written on the device
            if self._entry_type == _lib.TO_F32S:
                self._upload(prog.recs, schedule.rec_init_bytes(prog))
            self._upload(prog.params, Executable.counters(total_slices))
            self._upload(prog.accum, bytes(_lib.Accum()))
            if prog.host_accum is not None:
                ctypes.memset(prog.host_accum.data_ptr(), 0, ctypes.sizeof(_lib.Accum))
            return Executable(self, prog, total_slices, once)

    def _execute(self, tree, tables, num_groups, total_slices):
        exe = self._compile(tree, tables, num_groups, total_slices, once=True)
        try:
            return exe.run()
        finally:
            exe.close()

    def prepare(self, execution_plan, num_slice_limit=None):
        """Compile a sliced plan once; ``Executable.run()`` then contracts all of its
        slices with inputs already resident on the device."""
        total, tree, tables, groups = self._plan_inputs(execution_plan, num_slice_limit)
        return self._compile(tree, tables, groups, total)

    def _plan_inputs(self, execution_plan, num_slice_limit):
        """(slices, slice-free tree, leaf tables, groups) of a plan, as the batched executors
        take them (``jax_apis.py:253-313``): every leaf reordered to [slice row, unsliced
        axes] with its row lookup (``tensor_network.pyx:404-442``, ``tensor.py:95-119``).
        OR and variable leaves are described for the device to write (``device_leaves``);
        other leaves are built on the host."""
        network = execution_plan.network
        groups = [g for g in execution_plan.groups_to_slice if len(g) > 0]
        tree = network.remove_sliced_indices_from(execution_plan.tree, execution_plan.groups_to_slice)
        tables = {}
        if self._device_leaves:
            total, lookups = network.slice_lookups(execution_plan.groups_to_slice)
            for t, lookup in enumerate(lookups):
                spec_table = leaf_spec_table(network[t], lookup, len(groups))
                if spec_table is not None:
                    tables[t] = spec_table
        if len(tables) < len(network):
            total, sequences, _assignments = network.get_tensor_slices(execution_plan.groups_to_slice,
                                                                       self.create_tensor)
            for t, seq in enumerate(sequences):
                if t in tables:
                    continue
                reordered, lookup, shape = seq.reordered_tensor(self)
                reordered = np.asarray(reordered, dtype=np.float64)
                tables[t] = schedule.LeafTable(reordered.reshape(reordered.shape[0], -1), lookup, len(shape),
                                               copy=copy_weights(network[t]))
        if num_slice_limit is not None:
            total = min(total, int(num_slice_limit))
        return total, tree, tables, len(groups)

    def prepare_batch(self, plans):
        """Compile many unsliced plans into grouped schedules (``batch.compile_batch``),
        admitted in waves whose arenas fit the device budget (``mem_limit`` when set): the
        waves share one arena and run one after another.  Raises OutOfMemoryError when one
        instance alone does not fit (slice it first)."""
        from . import batch

        instances = []
        for plan in plans:
            total, tree, tables, groups = self._plan_inputs(plan, None)
            if groups:
                raise ValueError("prepare_batch takes unsliced plans")
            instances.append((tree, tables))
        budget = self._budget()
        per = fold.analyse_batch(instances, self._esize, self._regroup)
        folded = per is not None
        # instances are admitted by what their tensors take with one axis per edge, folded or
        # not (see choose_folded_batch); the analysis that gives it is needed only where all
        # of it at once might not fit
        bound = sum(schedule.peak_bound(tree, self._esize) + sum(t.size for t in tables.values()) * self._esize +
                    2048 * len(tables) for tree, tables in instances) if folded else None
        if folded and max(bound, sum(p["region"] + p["fixed"] for p in per)) <= budget:
            waves = [list(range(len(per)))] if per else []
        else:
            walk = batch.analyse_batch(instances, self._entry_type, regroup=self._regroup)
            if folded:
                for p, q in zip(per, walk):
                    q["region"] = max(q["region"], p["region"] + p["fixed"] - q["fixed"])
            else:
                per = walk
            waves = batch.admission_waves(walk, budget)
        if waves is None:
            raise OutOfMemoryError
        arena = self._alloc(max(max(batch.wave_arena_bytes(per, w) for w in waves), schedule.ALIGN))
        progs = []
        with self._settled():
            for w in waves:
                if folded:
                    prog = fold.compile_batch([per[i] for i in w], self._entry_type, self._alloc, arena, self._alloc_host)
                else:
                    prog = batch.compile_batch(None, self._entry_type, self._alloc, regroup=self._regroup,
                                               per=[per[i] for i in w], arena=arena)
                self._upload(prog.table, prog.table_host.tobytes())
                self._upload(prog.blob, prog.blob_host.tobytes())
                self._run(prog.build)  # OR / variable leaf tables written on the device
                if self._entry_type == _lib.TO_F32S:
                    self._upload(prog.recs, batch.rec_init_bytes(prog))
                progs.append(prog)
            return BatchExecutable(self, progs, arena)

    def contract_batch(self, plans):
        """Counts (floats) of many unsliced plans contracted together."""
        exe = self.prepare_batch(plans)
        try:
            res, _ = exe.run()
        finally:
            exe.close()
        return [r.value for r in res]

    def contract_sliced(self, execution_plan, num_slice_limit=None):
        total, tree, tables, groups = self._plan_inputs(execution_plan, num_slice_limit)
        if total <= 0:
            return 0
        return self._execute(tree, tables, groups, total).value

    def contract(self, network, contraction_tree):
        """Contract one network (sliced tensors keep size-1 axes, which are dropped)."""
        ctx = TreeContext()
        stack, tables = [], {}
        for node in contraction_tree.iterate_postorder():
            if node.is_leaf:
                t = node.tensor_index
                arr = np.asarray(network[t].build(self.create_tensor), dtype=np.float64)
                keep = [e for e, size in zip(node.free_edges, arr.shape) if size != 1]
                tables[t] = schedule.LeafTable(arr.reshape(1, -1), [], len(keep))
                stack.append(ctx.leaf_manual(t, keep))
            else:
                right = stack.pop()
                left = stack.pop()
                stack.append(ctx.join(left, right))
        res = self._execute(ctx.get_tree(stack[0]), tables, 0, 1)
        return np.array(res.value)

    # -- single join ---------------------------------------------------------------

    def _to_device(self, a):
        if isinstance(a, DeviceTensor):
            return a
        arr = np.asarray(a, dtype=np.float64)
        rec = None
        if self._entry_type == _lib.TO_F32S:
            m = float(np.max(np.abs(arr))) if arr.size else 0.0
            e = math.frexp(m)[1] if m > 0 else 0
            host = np.ldexp(arr, -e).astype(np.float32)
            r = _lib.ScaleRec(exp=e, maxbits=int(np.array([1.0], np.float32).view(np.uint32)[0]))
            rec = self._alloc(ctypes.sizeof(r))
            self._upload(rec, bytes(r))
        else:
            host = arr
        data = self._alloc(host.nbytes)
        self._upload(data, np.ascontiguousarray(host).tobytes())
        view = data[: host.nbytes].view(self._torch.float64 if host.dtype == np.float64 else self._torch.float32)
        return DeviceTensor(view, arr.shape, rec, self)

    def tensordot(self, a, b, axes):
        """``numpy.tensordot(a, b, axes)`` on the device; result keeps numpy's axis
        order (left free axes, then right free axes)."""
        for t in (a, b):
            if any(d != 2 for d in (t.shape if isinstance(t, DeviceTensor) else np.shape(t))):
                raise ValueError("HipAPI tensors must have all dimensions 2")
        try:
            return self._tensordot(self._to_device(a), self._to_device(b), list(axes[0]), list(axes[1]))
        except BaseException:
            self.synchronize()  # (see _settled, which would take 2 us of a small join)
            raise

    def _tensordot(self, A, B, lmap, rmap):
        g = schedule.join_geometry(A.rank, B.rank, lmap, rmap)
        g["var"] = schedule.choose_variant(g, 1, self._esize)
        out_rank = g["fx"] + g["fy"]
        out_shape = tuple(A.shape[i] for i in range(A.rank) if i not in lmap) + tuple(
            B.shape[i] for i in range(B.rank) if i not in rmap)
        cbuf = self._alloc((1 << out_rank) * self._esize)
        scaled = self._entry_type == _lib.TO_F32S
        crec = self._alloc(ctypes.sizeof(_lib.ScaleRec)) if scaled else None
        X, Y = (A, B) if g["x_is_left"] else (B, A)
        d = _lib.JoinDesc()
        d.x, d.y, d.c = X.data.data_ptr(), Y.data.data_ptr(), cbuf.data_ptr()
        if scaled:
            d.xs, d.ys, d.cs = X.rec.data_ptr(), Y.rec.data_ptr(), crec.data_ptr()
        d.fx, d.fy, d.s, d.shf, d.shy = g["fx"], g["fy"], g["s"], g["shf"], g["shy"]
        d.nbatch = 1
        d.xf_pos, d.xs_pos = schedule._pos_array(g["xf"]), schedule._pos_array(g["xs"])
        d.yf_pos, d.ys_pos = schedule._pos_array(g["yf"]), schedule._pos_array(g["ys"])
        v = g["var"]
        launches, blob = [], []
        if scaled:
            launches.append(_lib.Launch(op=_lib.TO_OP_SCALE_CLEAR, grid=1, aux0=crec.data_ptr(), iaux0=1))
        keep = [cbuf, crec]

        def launch(desc, **kw):  # a launch of one descriptor; all of them go up together
            launches.append(_lib.Launch(count=1, **kw))
            blob.append((launches[-1], bytes(desc)))

        if v["kind"] == "gemm":
            ops = []
            for need, T, fpos, spos in ((v["perm_x"], X, g["xf"], g["xs"]), (v["perm_y"], Y, g["yf"], g["ys"])):
                if not need:
                    ops.append(T.data.data_ptr())
                    continue
                out_pos = [0] * T.rank
                for t, p in enumerate(spos):
                    out_pos[p] = t
                for i, p in enumerate(fpos):
                    out_pos[p] = len(spos) + i
                dst = self._alloc((1 << T.rank) * self._esize)
                pd, grid, lds, pvar = schedule.perm_desc(T.data.data_ptr(), dst.data_ptr(), T.rank, out_pos, 1,
                                                         1 << T.rank, self._esize)
                launch(pd, op=_lib.TO_OP_PERMUTE, variant=pvar, grid=grid, lds=lds)
                keep.append(dst)
                ops.append(dst.data_ptr())
            gd = _lib.GemmDesc()
            gd.a, gd.b, gd.c = ops[0], ops[1], cbuf.data_ptr()
            gd.ldcm, gd.ldcn = 1 << g["shf"], 1 << g["shy"]
            if scaled:
                gd.as_, gd.bs, gd.cs = X.rec.data_ptr(), Y.rec.data_ptr(), crec.data_ptr()
            gd.mlog, gd.nlog, gd.klog = g["fx"], g["fy"], g["s"]
            gd.nbatch, gd.block0, gd.nblocks = 1, 0, v["nblocks"]
            launch(gd, op=_lib.TO_OP_GEMM, variant=v["tile"], grid=v["nblocks"])
        elif v["kind"] == "stream":
            d.nblocks, d.nych, d.nsplit = v["nblocks"], v["nych"], 1
            d.lnych = v["nych"].bit_length() - 1
            d.stage = int(v["stage"])
            launch(d, op=_lib.TO_OP_JOIN_STREAM, variant=schedule.stream_variant(v, g), grid=v["nblocks"], lds=v["lds"])
        else:
            part = self._alloc(v["nout"] * v["nsplit"] * 8)  # double partial sums
            d.partial = part.data_ptr()
            d.nsplit, d.nblocks = v["nsplit"], v["nblocks"]
            d2 = _lib.JoinDesc.from_buffer_copy(bytes(d))
            d2.nblocks = v["fin_blocks"]
            launch(d, op=_lib.TO_OP_JOIN_SPLITK, grid=v["nblocks"])
            launch(d2, op=_lib.TO_OP_JOIN_FINISH, variant=v["fin_variant"], grid=v["fin_blocks"])
            keep.append(part)
        table = self._alloc(sum(len(data) for _, data in blob))
        at = 0
        for L, data in blob:
            L.descs = table.data_ptr() + at
            at += len(data)
        self._upload(table, b"".join(data for _, data in blob))
        keep.append(table)
        self._run(launches)
        self.finish()
        tdtype = self._torch.float64 if not scaled else self._torch.float32
        view = cbuf[: (1 << out_rank) * self._esize].view(tdtype)
        return DeviceTensor(view, out_shape, crec, self)

    def permute(self, tensor, perm):
        """Device ``numpy.transpose`` of an all-dimension-2 tensor (returns numpy)."""
        with self._settled():
            return self._permute(self._to_device(tensor), perm)

    def _permute(self, A, perm):
        out = self._alloc((1 << A.rank) * self._esize)
        p = (ctypes.c_int32 * max(1, len(perm)))(*perm)
        rc = self._lib.to_permute(ctypes.c_void_p(A.data.data_ptr()), ctypes.c_void_p(out.data_ptr()), A.rank,
                                  ctypes.addressof(p), self._esize, 1, ctypes.c_void_p(self._stream.cuda_stream))
        _lib.check(rc, "to_permute")
        self.synchronize()
        tdtype = self._torch.float64 if self._esize == 8 else self._torch.float32
        view = out[: (1 << A.rank) * self._esize].view(tdtype)
        return DeviceTensor(view, tuple(A.shape[i] for i in perm), A.rec, self).numpy()


class HipF32API(HipAPI):
    """The FP32-scaled executor as its own library choice."""

    def __init__(self, device=0):
        super().__init__(device)
        self._entry_type = _lib.TO_F32S


HIP_APIS = {"hip": HipAPI, "hip-f32": HipF32API}
