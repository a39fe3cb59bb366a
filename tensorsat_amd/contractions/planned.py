"""
Planned (tree) contractions: the counterpart of the reference's ``CotengraContraction``
(``tensorsat/contractions/cotengra.py:52-131``) with this package's planner in place of
cotengra.

Construction plans a binary tree over the wiring's hypergraph (``optimize``: ``"greedy"``,
``"hyper"``, ``"elim"`` or ``"auto"``, the cheapest of elimination-order and hyper-greedy
trees by the cotengra cost model), optionally slicing wires down to a size target.
``contract`` walks the tree calling the box class's pairwise contraction per node, as
cotengra's ``ContractionTree.contract`` does through ``_autoray.einsum`` (a wire is
summed at the first node after which no other tensor and no out port holds it), OR-s
(``+``) the slices, adds dangling out wires and rewires to the out wires.
Small trees over host leaves run as one device job instead (:class:`SmallTree`: the same steps
in one launch).
:meth:`contract_program` compiles the whole tree for the device executor instead.
"""

from __future__ import annotations

import itertools

import numpy as np

from .. import _native
from .. import plan as _plan
from .. import program as _prog
from ..network import Diagram, Wiring
from ..rel import DeviceRel
from .abc import Contraction


def plan_wiring(wiring: Wiring, optimize: str = "auto", *, trials: int = 32, seed: int = 0) -> _plan.Plan:
    if optimize == "greedy":
        return _plan.greedy(wiring)
    if optimize == "hyper":
        return _plan.hyper(wiring, trials=trials, seed=seed)
    if optimize == "elim":
        p = _prog.elim(wiring, trials=max(1, trials // 4), seed=seed)
        p.cost = _plan.tree_cost(wiring, p)
        return p
    if optimize in ("auto", "auto-hq"):
        cands = [_plan_elim(wiring, trials, seed), _plan.hyper(wiring, trials=trials, seed=seed)]
        for c in cands:
            c.cost = _plan.tree_cost(wiring, c)
        return min(cands, key=lambda p: (p.cost.log2_max_size, p.cost.log2_flops))
    raise ValueError(f"unknown optimize {optimize!r}")


def _plan_elim(wiring: Wiring, trials: int, seed: int) -> _plan.Plan:
    return _prog.elim(wiring, trials=max(1, trials // 4), seed=seed)


def tree_steps(wiring: Wiring, path: np.ndarray, drop=()):
    """
    Per merge: (lhs id, rhs id, lhs wires, rhs wires, out wires) under the merge rule,
    with wires in ``drop`` (sliced) removed everywhere.  Out wires keep lhs order then
    rhs-only order.
    """
    drop = set(drop)
    S = wiring.num_slots
    legs: list[list[int]] = []
    count: dict[int, int] = {}
    for ws in wiring.slot_wires_list:
        u = []
        for w in ws:
            if w not in drop and w not in u:
                u.append(w)
        legs.append(u)
        for w in u:
            count[w] = count.get(w, 0) + 1
    for w in set(wiring.out_wires):
        count[w] = count.get(w, 0) + 1
    steps = []
    for a, b in path.tolist():
        la, lb = legs[a], legs[b]
        sb = set(lb)
        out = []
        for w in la + [w for w in lb if w not in set(la)]:
            c = (w in set(la)) + (w in sb)
            if count.get(w, 0) > c:
                out.append(w)
        for w in la:
            count[w] -= 1
        for w in lb:
            count[w] -= 1
        for w in out:
            count[w] = count.get(w, 0) + 1
        legs.append(out)
        steps.append((a, b, la, lb, out))
    root_legs = legs[-1] if legs else []
    return steps, root_legs


class SmallTree:
    """
    A whole tree as one device job (``ts_program_run_small``): its step records, laid out
    once per contraction, and where each leaf entry of a diagram goes in the job's leaves.
    The steps are the tree's (:func:`tree_steps`), so every intermediate has the values that
    the walk gives it, in the compiler's layouts; the result is in out-wire order.
    """

    # Products per step above which a workgroup's 256 lanes are no longer ahead of a launch
    # per step: a step of 2^14 products takes them about 4 us, the walk 35 us of host.
    MAX_TERMS = 1 << 14

    @staticmethod
    def slot_shapes(wiring: Wiring, tree: _plan.Plan) -> list[tuple[int, ...]] | None:
        """The leaves' shapes; None where the wiring or the tree has to take the walk: sliced
        trees, extents other than 2, repeated or dangling wires, a single slot, or leaves that
        do not fit one workgroup."""
        slots, outs = wiring.slot_wires_list, wiring.out_wires
        if len(slots) < 2 or len(tree.sliced) or any(d != 2 for d in wiring.wire_dims):
            return None
        held = {w for ws in slots for w in ws}
        if len(set(outs)) != len(outs) or not held.issuperset(outs) or any(len(set(ws)) != len(ws) for ws in slots):
            return None
        if sum(1 << len(ws) for ws in slots) > _native.SMALL_LEAVES:
            return None
        return [(2,) * len(ws) for ws in slots]

    @classmethod
    def build(cls, wiring: Wiring, tree: _plan.Plan, shapes=None) -> "SmallTree | None":
        """None where the walk has to run (:meth:`slot_shapes`, or tensors that do not fit one
        workgroup)."""
        shapes = shapes or cls.slot_shapes(wiring, tree)
        if shapes is None or _plan.tree_cost(wiring, tree).log2_max_size > 15:
            return None
        # The compiler lays leaf entries out in its own order: compiled with each entry's
        # index (its low, then its high byte) as the value, the leaves say which goes where.
        sizes = [1 << len(shape) for shape in shapes]
        index = np.split(np.arange(sum(sizes)), np.cumsum(sizes)[:-1])

        def compiled(shift: int) -> _prog.Program:
            return _prog.compile_network(wiring, [((ix >> shift) & 255).astype(np.uint8) for ix in index], tree)

        lo = compiled(0)
        terms = np.ldexp(1.0, lo.steps["out_rank"].astype(int) + lo.steps["sum_rank"]).sum()
        if (len(lo.jobs) != 1 or int(lo.jobs["arena_elems"][0]) > _native.SMALL_ARENA or
                lo.leaves.size > _native.SMALL_LEAVES or terms > cls.MAX_TERMS * len(lo.steps)):
            return None
        high = compiled(8).leaves.astype(np.int64) << 8 if sum(sizes) > 256 else 0
        self = object.__new__(cls)
        self.prog = lo
        self.source = lo.leaves.astype(np.int64) | high
        self.shapes = shapes
        self.rank = len(wiring.out_wires)
        self.device_steps = {}
        return self

    @staticmethod
    def entries(shapes, blocks) -> np.ndarray | None:
        """All leaf entries in slot order, or None if the blocks are not 0/1 host arrays of the
        slots' shapes."""
        if not all(type(b) is np.ndarray for b in blocks) or [b.shape for b in blocks] != shapes:
            return None
        flat = np.concatenate([b.reshape(-1) for b in blocks])
        return flat if flat.dtype == np.uint8 and flat.max() <= 1 else None

    def leaf_bits(self, blocks) -> np.ndarray | None:
        """The job's leaves as bits, or None where :meth:`entries` is."""
        flat = self.entries(self.shapes, blocks)
        return None if flat is None else self.pack(flat)

    def pack(self, flat: np.ndarray) -> np.ndarray:
        return np.packbits(flat[self.source], bitorder="little")

    def run(self, bits: np.ndarray, box_class, mode: str):
        import torch

        N = _native
        L = N.lib()
        dev = torch.cuda.current_device()
        stream = torch.cuda.current_stream()
        held = self.device_steps.get(dev)
        if held is None:  # a synchronous upload: complete for every stream
            held = torch.from_numpy(self.prog.steps.view(np.uint8)).cuda(), stream.cuda_stream
            self.device_steps[dev] = held
        steps, owner = held
        if owner != stream.cuda_stream:  # not given back while this stream still reads it
            steps.record_stream(stream)
        res = torch.empty(max(16, 1 << self.rank), dtype=torch.uint8, device="cuda")
        N.check(L.ts_program_run_small(N.host_ptr(self.prog.jobs), N.host_ptr(self.prog.steps), N.dptr(steps),
                                       N.host_ptr(bits), N.dptr(res), N.MODES[mode], N.stream_ptr()),
                "ts_program_run_small")
        return box_class._new(res, (2,) * self.rank)


class PlannedContraction(Contraction):
    """A contraction along a planned binary tree (``CotengraContraction`` counterpart)."""

    _small = False  # SmallTree or None, built on the first contraction of 0/1 host leaves

    def __getstate__(self):
        return {k: v for k, v in self.__dict__.items() if k != "_small"}  # holds device memory

    def __init__(self, box_class: type, wiring: Wiring, *, optimize: str = "auto",
                 slicing_target: float | None = None, trials: int = 32, seed: int = 0,
                 canonicalize: bool = True, sort_contraction_indices: bool = False) -> None:
        super().__init__(box_class, wiring)
        if wiring.num_wires == 0:
            raise ValueError("Cannot define contraction for empty wiring.")
        tree = plan_wiring(wiring, optimize, trials=trials, seed=seed)
        if slicing_target is not None and tree.cost is not None and tree.cost.log2_max_size > slicing_target:
            tree = _plan.slice_plan(wiring, tree, slicing_target, reconfigure_trials=trials, seed=seed)
        self._tree = tree

    @property
    def tree(self) -> _plan.Plan:
        return self._tree

    @property
    def path(self) -> tuple[tuple[int, int], ...]:
        return tuple(self._tree.linear_path())

    def _contract_boxes(self, boxes: list, fixed: dict[int, int]):
        cls = self.box_class
        wiring = self.wiring
        leaves = []
        for b, ws in zip(boxes, wiring.slot_wires_list):
            if fixed and any(w in fixed for w in ws):
                idx = tuple(fixed[w] if w in fixed else slice(None) for w in ws)
                # a sliced wire repeated within one slot is fixed on each of its ports
                b = b[idx]
            leaves.append(b)
        live = {}
        lw = {}
        for s, (b, ws) in enumerate(zip(leaves, wiring.slot_wires_list)):
            ws = [w for w in ws if w not in fixed]
            # repeated wires within one slot: take the diagonal first
            uniq = list(dict.fromkeys(ws))
            if len(uniq) != len(ws):
                b = cls._contract2(b, ws, cls.scalar(True), [], uniq)
            live[s] = b
            lw[s] = uniq
        steps, root = tree_steps(wiring, self._tree.path, fixed)
        S = wiring.num_slots
        for k, (a, b, la, lb, out) in enumerate(steps):
            res = cls._contract2(live.pop(a), lw.pop(a), live.pop(b), lw.pop(b), out)
            live[S + k] = res
            lw[S + k] = out
        if S == 0:
            box, wires = cls.scalar(True), []
        else:
            (key,) = live.keys()
            box, wires = live[key], list(lw[key])
            # a single slot: sum the wires that are not out wires
            keep = [w for w in wires if w in set(wiring.out_wires)]
            if keep != wires:
                box = box._rewire([wires.index(w) for w in keep])
                wires = keep
        dangling = [w for w in dict.fromkeys(wiring.out_wires) if w not in wires and w not in fixed]
        if dangling:
            box = cls.prod([box] + [cls.spider(wiring.wire_dims[w], 1) for w in dangling])
            wires = wires + dangling
        return box, wires

    def _small_bits(self, blocks) -> np.ndarray | None:
        """The leaves as bits of the tree's small job, or None where the walk runs.  The job is
        laid out (two compilations, a few ms) only for leaves that it takes."""
        small = self._small
        if small is None:
            return None
        shapes = small.shapes if small else SmallTree.slot_shapes(self.wiring, self._tree)
        flat = SmallTree.entries(shapes, blocks) if shapes else None
        if flat is None:
            return None
        if small is False:
            small = self._small = SmallTree.build(self.wiring, self._tree, shapes)
        return None if small is None else small.pack(flat)

    def contract(self, diagram: Diagram, *, order=None, autojit="auto", progbar: bool = False):
        """Validate and contract (``cotengra.py:100-128``)."""
        self.validate(diagram)
        if self.box_class is DeviceRel:
            bits = self._small_bits(diagram.blocks)
            if bits is not None:
                return self._small.run(bits, DeviceRel, DeviceRel._mode)
        boxes = self._boxes(diagram)
        sliced = list(self._tree.sliced)
        dims = self.wiring.wire_dims
        result = None
        wires_out = None
        for vals in itertools.product(*(range(dims[w]) for w in sliced)):
            box, wires = self._contract_boxes(boxes, dict(zip(sliced, vals)))
            result = box if result is None else result + box
            wires_out = wires
        out_wires = list(self.wiring.out_wires)
        if wires_out != out_wires:
            result = result._rewire([wires_out.index(w) for w in out_wires])
        return result

    def contract_program(self, diagram: Diagram) -> _prog.Program:
        """
        Compile the tree with the diagram's host leaves for the device step executors:
        one job, or with sliced wires one job per slice (the sliced wires fixed in every
        leaf that holds them, ``Box.__getitem__``; the jobs' results are to be OR-ed, or
        summed when counting).  Every job has the tree's steps with the sliced wires
        removed, in the compiler's layouts (contracted wires innermost in both operands,
        so dense steps take the MFMA route).  Needs extent-2 wires, unique wires per slot
        and a scalar result.
        """
        self.validate(diagram)
        if self.wiring.out_wires:
            raise NotImplementedError("compiled programs of sliced trees need a scalar result")
        leaves = [np.asarray(getattr(b, "tensor", b), dtype=np.uint8) for b in diagram.blocks]
        sliced = list(self._tree.sliced)
        if not sliced:
            return _prog.compile_network(self.wiring, leaves, self._tree)
        progs = _prog.compile_sliced(self.wiring, leaves, self._tree, sliced)
        return _prog.concat(progs, [np.zeros(1, np.int64)] * len(progs), 1)

    def __repr__(self) -> str:
        return "<PlannedContraction>"
