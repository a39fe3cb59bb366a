"""
Trees that run as one device job (host leaves, every tensor in one workgroup's LDS) against
the walk node by node and the oracle, and the diagrams that have to take the walk.
"""

import pickle

import numpy as np
import pytest

from oracle_box import OracleRel
from tensorsat_amd.contractions import PlannedContraction
from tensorsat_amd.contractions.planned import SmallTree
from tensorsat_amd.network import Diagram, Wiring
from tensorsat_amd.sat import CNFInstance


def _cnf_diagram(n, ratio, seed, inputs=None):
    cnf = CNFInstance.random(3, n, int(round(ratio * n)), rng=seed)
    return (cnf.inputs("_" * n if inputs is None else inputs) >> cnf.diagram()).flatten()


def _random_diagram(rng, slots, wires, outs, rank=4):
    ws = [[int(w) for w in rng.choice(wires, size=int(rng.integers(1, rank + 1)), replace=False)] for _ in range(slots)]
    held = sorted({w for s in ws for w in s})
    out = [int(w) for w in rng.permutation(held)[:outs]]
    blocks = [(rng.random((2,) * len(s)) < 0.8).astype(np.uint8) for s in ws]
    return Diagram(Wiring([2] * wires, ws, out), blocks)


def test_trees_that_take_the_walk():
    rng = np.random.default_rng(0)
    leaf = np.ones((2, 2), np.uint8)

    def small(*args, **kw):
        w = Wiring(*args)
        c = PlannedContraction(OracleRel, w, **kw)
        return SmallTree.build(w, c.tree)

    assert small([2] * 3, [[0, 1], [1, 2]], [0, 2]) is not None
    assert small([3] * 3, [[0, 1], [1, 2]], [0, 2]) is None  # extents
    assert small([2] * 3, [[0, 1, 2]], [0]) is None  # one slot
    assert small([2] * 3, [[0, 0], [0, 1]], [1]) is None  # repeated wire in a slot
    assert small([2] * 3, [[0, 1], [1, 2]], [0, 0]) is None  # repeated out wire
    assert small([2] * 4, [[0, 1], [1, 2]], [3, 0]) is None  # dangling out wire
    assert small([2] * 20, [[*range(0, 12)], [*range(8, 20)]], [*range(20)]) is None  # too large a result
    t = small([2] * 3, [[0, 1], [1, 2]], [0, 2])
    assert t.leaf_bits([leaf, leaf]) is not None
    assert t.leaf_bits([leaf, leaf[0]]) is None and t.leaf_bits([leaf, 2 * leaf]) is None
    assert t.leaf_bits([leaf, leaf.tolist()]) is None and t.leaf_bits([leaf, leaf.astype(np.int64)]) is None
    # every leaf entry lands where the compiler puts it
    d = _random_diagram(rng, 9, 8, 3)
    s = SmallTree.build(d.wiring, PlannedContraction(OracleRel, d.wiring).tree)
    from tensorsat_amd import program as PG

    prog = PG.compile_network(d.wiring, list(d.blocks), PlannedContraction(OracleRel, d.wiring).tree)
    assert (s.prog.steps == prog.steps).all()
    got = np.unpackbits(s.leaf_bits(d.blocks), bitorder="little")[: prog.leaves.size]
    for st in prog.steps:
        for off, rank in ((st["lhs_off"], st["lhs_rank"]), (st["rhs_off"], st["rhs_rank"])):
            if off < prog.jobs["num_leaf_bytes"][0] and off not in prog.steps["out_off"]:
                assert (got[off : off + (1 << rank)] == prog.leaves[off : off + (1 << rank)]).all()


def test_jobs_are_laid_out_for_host_leaves_only(monkeypatch):
    """Leaves that take the walk never reach the compiler."""
    from tensorsat_amd.rel import DeviceRel

    leaf, wide = np.ones((2, 2), np.uint8), np.ones((2,) * 15, np.uint8)
    for wires, blocks in (
        ([[0, 1], [1, 2]], [leaf, object()]), ([[0, 1], [1, 2]], [object(), object()]),
        ([[0, 1], [1, 2]], [leaf, 2 * leaf]), ([[0, 1], [1, 2]], [leaf.astype(bool)] * 2),
        ([[0, 1], [1, 2]], [leaf, leaf[0]]), ([[*range(15)], [*range(1, 16)]], [wide, wide]),
    ):
        w = Wiring([2] * (1 + max(max(ws) for ws in wires)), wires, [0])
        c = PlannedContraction(DeviceRel, w)
        monkeypatch.setattr(SmallTree, "build", lambda *a: pytest.fail("laid out"))
        assert c._small_bits(blocks) is None and c._small is False
        monkeypatch.undo()
        host = [np.ones((2,) * len(ws), np.uint8) for ws in wires]
        bits = c._small_bits(host)  # 2^16 leaf entries are too many
        assert (bits is None) == (len(wires[0]) == 15) and (c._small is False) == (bits is None)


def _walk(wiring, tree, blocks, mode):
    """The tree's steps one by one in numpy, the result in out-wire order."""
    from tensorsat_amd.contractions.planned import tree_steps

    live = {i: (b.astype(np.int64), list(ws)) for i, (b, ws) in enumerate(zip(blocks, wiring.slot_wires_list))}
    for k, (a, b, _, _, out) in enumerate(tree_steps(wiring, tree.path)[0]):
        (x, lx), (y, ly) = live.pop(a), live.pop(b)
        ids = {w: i for i, w in enumerate(dict.fromkeys(lx + ly))}
        cnt = np.einsum(x, [ids[w] for w in lx], y, [ids[w] for w in ly], [ids[w] for w in out])
        live[wiring.num_slots + k] = (cnt % 256 if mode == "MOD256" else cnt).astype(bool).astype(np.int64), list(out)
    ((r, ws),) = live.values()
    return r.transpose([ws.index(w) for w in wiring.out_wires]).reshape(-1)


@pytest.mark.parametrize("mode", ["GT0", "MOD256"])
def test_job_equals_the_walk_on_any_wiring(mode):
    """The job's records and leaves, run by the oracle: scalar slots, unheld wires, wires summed
    in one slot, unconnected parts, any out order."""
    from oracle import executor as OX
    from tensorsat_amd import program as PG

    rng, taken = np.random.default_rng(3), 0
    for i in range(200):
        n = int(rng.integers(1, 14))
        ws = [[int(w) for w in rng.choice(n, size=min(n, int(rng.integers(0, 6))), replace=False)]
              for _ in range(int(rng.integers(2, 14)))]
        held = sorted({w for s in ws for w in s})
        w = Wiring([2] * n, ws, [int(x) for x in rng.permutation(held)[: int(rng.integers(0, 7))]])
        blocks = [np.asarray(rng.random((2,) * len(s)) < (0.95 if i % 3 else 1.1)).astype(np.uint8).reshape((2,) * len(s))
                  for s in ws]
        c = PlannedContraction(OracleRel, w)
        t = SmallTree.build(w, c.tree)
        if t is None:
            continue
        taken += 1
        leaves = np.unpackbits(t.leaf_bits(blocks), bitorder="little")[: t.prog.leaves.size]
        got, _ = OX.run_job(PG.Program(t.prog.jobs, t.prog.steps, leaves, t.prog.stats, {}), 0, mode)
        np.testing.assert_array_equal(np.asarray(got).reshape(-1), _walk(w, c.tree, blocks, mode), err_msg=f"{ws}")
    assert taken > 150


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["GT0", "MOD256"])
def test_small_trees_match_the_walk_and_the_oracle(mode):
    from tensorsat_amd.rel import DeviceRel

    rng = np.random.default_rng(7)
    diagrams = [_cnf_diagram(n, r, n) for n, r in ((3, 1.0), (6, 2.0), (9, 3.0), (10, 3.5), (12, 3.5), (14, 2.0))]
    diagrams += [_cnf_diagram(12, 4.0, 5, inputs="0" * 12)]  # scalar result
    diagrams += [_random_diagram(rng, int(rng.integers(2, 40)), int(rng.integers(4, 24)), int(rng.integers(0, 6)))
                 for _ in range(25)]
    # 2^10 terms in one step: counts of 0 mod 256
    diagrams.append(Diagram(Wiring([2] * 12, [[*range(11)], [*range(10), 11]], [11, 10]),
                            [np.ones((2,) * 11, np.uint8)] * 2))
    # 16384 leaf entries and a result of 2^15: an arena of 48 KB
    wide = [[*range(13)], [*range(2, 13), 13, 14], [0], [14]]
    diagrams.append(Diagram(Wiring([2] * 15, wide, [*range(14, -1, -1)]),
                            [(rng.random((2,) * len(ws)) < 0.7).astype(np.uint8) | (len(ws) == 1) for ws in wide]))
    with DeviceRel.mode_scope(mode):
        for i, d in enumerate(diagrams):
            c = PlannedContraction(DeviceRel, d.wiring)
            print(f"{mode} diagram {i}: {d.wiring.num_slots} slots, {len(d.wiring.out_wires)} out", flush=True)
            first, again = c.contract(d), c.contract(d)
            assert c._small is not None
            c._small = None  # the walk
            walk = c.contract(d)
            assert first.tensor_shape == walk.tensor_shape
            np.testing.assert_array_equal(first.tensor, walk.tensor)
            np.testing.assert_array_equal(again.tensor, walk.tensor)
            if mode == "GT0":
                np.testing.assert_array_equal(walk.tensor,
                                              PlannedContraction(OracleRel, d.wiring).contract(d).tensor)


def _wide_tree(rng):
    """28672 leaf entries at most and a result of 2^15: an arena of 65056 of 65536 entries."""
    ws = [[8, 3], [9, 0], [11, 0, 12, 6, 4, 8, 15, 10], [1, 9, 4, 14, 13, 7, 8, 0, 6, 15, 5, 3, 10],
          [7, 13, 6, 0, 10, 15, 12, 2, 5, 11, 8], [13, 14, 1, 7, 10, 11, 9, 4]]
    out = [13, 9, 4, 1, 3, 14, 0, 7, 6, 11, 15, 10, 5, 8, 12]
    return Diagram(Wiring([2] * 16, ws, out), [(rng.random((2,) * len(s)) < 0.9).astype(np.uint8) for s in ws])


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["GT0", "MOD256"])
def test_largest_arenas(mode):
    """Up to the 65536 entries of LDS that a job may take; one more is refused."""
    import torch

    from tensorsat_amd import _native as N
    from tensorsat_amd.rel import DeviceRel

    d = _wide_tree(np.random.default_rng(8))
    c = PlannedContraction(DeviceRel, d.wiring)
    want = _walk(d.wiring, c.tree, d.blocks, mode)
    with DeviceRel.mode_scope(mode):
        np.testing.assert_array_equal(c.contract(d).tensor.reshape(-1), want)
    small = c._small
    assert small is not None and int(small.prog.jobs["arena_elems"][0]) > 65000
    steps, bits = torch.from_numpy(small.prog.steps.view(np.uint8)).cuda(), small.leaf_bits(d.blocks)
    for elems in (65536, 65537):
        job = small.prog.jobs.copy()
        job["arena_elems"] = elems
        res = torch.full((1 << 15,), 7, dtype=torch.uint8, device="cuda")
        print(f"{mode}: {elems} arena entries", flush=True)
        rc = N.lib().ts_program_run_small(N.host_ptr(job), N.host_ptr(small.prog.steps), N.dptr(steps), N.host_ptr(bits),
                                          N.dptr(res), N.MODES[mode], N.stream_ptr())
        assert rc == (0 if elems == 65536 else N.TS_EUNSUPPORTED)
        np.testing.assert_array_equal(res.cpu().numpy(), want if rc == 0 else np.full(1 << 15, 7))


@pytest.mark.gpu
def test_device_blocks_and_other_streams():
    import torch

    from tensorsat_amd.rel import DeviceRel

    d = _cnf_diagram(8, 3.0, 1)
    c = PlannedContraction(DeviceRel, d.wiring)
    want = c.contract(d).tensor
    boxes = Diagram(d.wiring, [DeviceRel(np.asarray(b)) for b in d.blocks])
    np.testing.assert_array_equal(c.contract(boxes).tensor, want)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        other = c.contract(d)
    s.synchronize()
    np.testing.assert_array_equal(other.tensor, want)
    copied = pickle.loads(pickle.dumps(c))  # a saved plan holds no device memory
    assert copied._small is False
    np.testing.assert_array_equal(copied.contract(d).tensor, want)
