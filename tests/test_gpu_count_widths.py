"""
Counting with narrow storage: the widths written into the step records (CPU), and exact counts
on the GPU at the edges of uint32 and uint64 (products of disjoint clauses have closed forms).
"""

import numpy as np
import pytest

from oracle import brute
from tensorsat_amd import program as PG
from tensorsat_amd.network import Wiring
from tensorsat_amd.sat import CNFInstance

OUT32, EXACT = 16, 32


def _bounds(prog, job):
    """(bound bits, lhs kind, rhs kind) per step of a job, by following arena offsets."""
    held = {}
    for st in prog.steps[job["step_begin"] : job["step_begin"] + job["num_steps"]]:
        sides = [int(st["lhs_off"])] + ([] if st["flags"] & PG.STEP_NORHS else [int(st["rhs_off"])])
        parts = [held.get(o, (0, 2)) for o in sides]
        b = sum(p[0] for p in parts) + int(st["sum_rank"])
        yield b, parts[0][1], parts[1][1] if len(parts) > 1 else 0
        held[int(st["out_off"])] = (b, 1 if b <= 31 else 0)


def _check_tags(prog):
    got = PG.count_widths(prog)
    seen = set()
    for job in got.jobs:
        steps = got.steps[job["step_begin"] : job["step_begin"] + job["num_steps"]]
        last = [int(o) for o in steps["out_off"]]
        final = len(last) - 1 - last[::-1].index(int(job["result_off"])) if int(job["result_off"]) in last else -1
        for i, (st, (b, kl, kr)) in enumerate(zip(steps, _bounds(prog, job))):
            want = kl | kr << 2 | (EXACT if b <= 63 else 0) | (OUT32 if b <= 31 and i != final else 0)
            assert int(st["pad"][0]) == want, (i, b)
            seen.add(want & (OUT32 | EXACT))
    assert not prog.steps["pad"].any()  # the given program is left alone
    return seen


def _disjoint(m):
    """m clauses on 3 variables each, as one job: 7^m models, 3 m summed bits."""
    w = Wiring([2] * (3 * m), [[3 * i, 3 * i + 1, 3 * i + 2] for i in range(m)], [])
    leaf = np.ones((2, 2, 2), np.uint8)
    leaf[1, 0, 1] = 0
    return PG.compile_network(w, [leaf] * m, PG.elim(w, trials=1))


def test_widths_follow_the_summed_bits():
    cnfs = [CNFInstance.random(3, n, 3 * n, rng=n) for n in (12, 30, 44)]
    assert _check_tags(PG.sat_batch(cnfs, width=10)) == {OUT32 | EXACT, EXACT}
    for m, kinds in ((10, {OUT32 | EXACT, EXACT}), (21, {OUT32 | EXACT, EXACT}), (23, {OUT32 | EXACT, EXACT, 0})):
        assert _check_tags(_disjoint(m)) == kinds


def test_leaf_bytes_above_one_and_shared_records():
    w = Wiring([2] * 3, [[0, 1], [1, 2]], [])
    prog = PG.compile_network(w, [np.ones((2, 2), np.uint8)] * 2, PG.elim(w, trials=1))
    narrow = PG.count_widths(prog).steps["pad"][:, 0]
    prog.leaves[0] = 200  # 8 bits per leaf: 16 + 3 summed
    assert (PG.count_widths(prog).steps["pad"][:, 0] == narrow).all()
    two = PG.concat([prog], [np.zeros(1, np.int64)], 1)
    two.jobs = np.concatenate([two.jobs, two.jobs])  # both jobs run the same records
    assert not PG.count_widths(two).steps["pad"].any()


@pytest.mark.gpu
def test_counts_at_the_edges_of_the_widths():
    from tensorsat_amd.executor import BatchCounter

    for m in (1, 9, 10, 11, 20, 21, 22):  # 7^22 < 2^62, a bound of 66 bits: checked arithmetic
        assert BatchCounter(_disjoint(m)).run() == [7**m], m
    with pytest.raises(OverflowError):
        BatchCounter(_disjoint(23)).run()  # 7^23 > 2^64


@pytest.mark.gpu
@pytest.mark.parametrize("n,width", [(14, 3), (20, 9), (22, 12), (24, 16)])
def test_counts_match_brute_force(n, width):
    from tensorsat_amd.executor import BatchCounter

    cnfs = [CNFInstance.random(3, n, int(r * n), rng=40 * n + i) for i, r in enumerate((1.0, 2.0, 3.0))]
    got = BatchCounter(PG.sat_batch(cnfs, width=width)).run()
    assert got == [brute.count(c.num_vars, c.clauses) for c in cnfs]


@pytest.mark.gpu
def test_wide_sums_and_general_steps():
    """A step of 2 out bits that is not K-innermost, and one summing 8 bits at once."""
    from tensorsat_amd.executor import BatchCounter
    from wide_steps import wide_sum_program

    for permute in (True, False):
        prog, leaves = wide_sum_program(3, out_wires=(), n=10, density=0.5, permute=permute)
        got = BatchCounter(prog).run()
        off = [int(prog.steps["lhs_off"][0]), int(prog.steps["rhs_off"][0])]
        lhs, rhs = (prog.leaves[o : o + 1024].astype(np.int64) for o in off)
        idx = np.arange(1024)
        at = [np.zeros(1024, np.int64), np.zeros(1024, np.int64)]
        for k in range(10):
            for side, name in enumerate(("c_lpos", "c_rpos")):
                at[side] |= ((idx >> k) & 1) << int(prog.steps[name][0, k])
        assert got == [int((lhs[at[0]] * rhs[at[1]]).sum())]


def _steps_by_hand(kind):
    """128 leaf entries of ones, tensors written over them, one operand (or the result) that is a
    part of a tensor; and the count."""
    copy = lambda lhs, rank, out: (lhs, out, rank, rank)
    total = lambda lhs, rank, out: (lhs, out, rank, 0)
    rows = {
        # the upper half of a tensor of 32 at 32
        "upper half": [copy(0, 5, 32), total(48, 4, 128)],
        # a tensor at 48, then a larger one over it, whose upper half is read there
        "overwritten": [copy(0, 4, 48), copy(0, 5, 32), total(48, 4, 128)],
        # the lower half of a tensor whose upper half was overwritten
        "remains": [copy(0, 5, 32), copy(0, 4, 48), total(32, 4, 128)],
        # the result is the middle entry of a tensor
        "result": [copy(0, 5, 112)],
        "whole": [copy(0, 4, 32), copy(0, 4, 48), total(48, 4, 128)],
    }[kind]
    steps = np.zeros(len(rows), PG.STEP_DTYPE)
    for name in ("o_lpos", "o_rpos", "c_lpos", "c_rpos"):
        steps[name] = PG.NOPOS
    for st, (lhs, out, rank, ro) in zip(steps, rows):
        st["lhs_off"], st["rhs_off"], st["out_off"] = lhs, lhs, out
        st["lhs_rank"], st["out_rank"], st["sum_rank"] = rank, ro, rank - ro
        st["flags"] = PG.STEP_NORHS | PG.STEP_KINNER
        st["o_lpos"][:ro] = range(ro)
        st["c_lpos"][: rank - ro] = range(rank - ro)
    jobs = np.zeros(1, PG.JOB_DTYPE)
    jobs["num_steps"], jobs["num_leaf_bytes"], jobs["result_off"], jobs["arena_elems"] = len(rows), 128, 128, 160
    want = 1 if kind == "result" else 16
    return PG.Program(jobs, steps, np.ones(128, np.uint8), np.zeros((1, PG.NSTAT), np.int64), {}), want


@pytest.mark.parametrize("kind", ["upper half", "overwritten", "remains", "result", "whole"])
def test_parts_of_tensors_stay_uint64(kind):
    prog, _ = _steps_by_hand(kind)
    PG.validate(prog)
    got = PG.count_widths(prog).steps
    if kind == "whole":
        assert [int(t) for t in got["pad"][:, 0]] == [2 | OUT32 | EXACT, 2 | OUT32 | EXACT, 1 | EXACT]
    else:
        assert not got["pad"].any() and not (got["flags"] & PG.STEP_WIDTHS).any()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["upper half", "overwritten", "remains", "result", "whole"])
def test_counts_over_parts_of_tensors(kind):
    from tensorsat_amd.executor import BatchCounter

    prog, want = _steps_by_hand(kind)
    for widths in (True, False, None):
        assert BatchCounter(prog, widths=widths).run() == [want]


def _packet_programs():
    for width, sizes in ((6, (12, 20, 30)), (4, (16, 22, 24))):
        yield PG.sat_batch([CNFInstance.random(3, n, 3 * n, rng=n) for n in sizes], width=width)


def test_widths_and_lanes_exclude_each_other():
    for prog in _packet_programs():
        pk = PG.packetize(prog)
        assert (pk.steps["pad"][:, 0] > 0).any()  # lanes
        wide = PG.count_widths(pk)
        assert not (wide.steps["flags"] & (PG.STEP_PACKET | PG.STEP_PEND)).any()
        assert (wide.steps["flags"] & PG.STEP_WIDTHS).all() and "packetized" not in wide.meta
        with pytest.raises(ValueError):
            PG.lanes(wide)
        assert (pk.steps["flags"] & PG.STEP_PACKET).all()  # the given program is left alone
        again = PG.packetize(PG.count_widths(prog))
        assert not (again.steps["flags"] & PG.STEP_WIDTHS).any()
        assert (again.steps == pk.steps).all()
        PG.lanes(again)


@pytest.mark.gpu
def test_records_without_widths_count_as_uint64():
    """Packet-form records (pad[0] = a lane) and records whose pad was never cleared, through
    both C entries."""
    from tensorsat_amd.executor import BatchCounter, DeviceProgram

    for prog in _packet_programs():
        want = BatchCounter(prog).run()
        dirty = PG.Program(prog.jobs, prog.steps.copy(), prog.leaves, prog.stats, {})
        dirty.steps["pad"] = np.random.default_rng(0).integers(0, 256, dirty.steps["pad"].shape)
        for other in (PG.packetize(prog), dirty):
            counter = BatchCounter(other, widths=True)
            counter.dp = DeviceProgram(other)  # the records as they are
            for counter.widths in (True, False):  # ts_batch_count_widths, ts_batch_count
                assert counter.run() == want


def test_tags_are_the_widths():
    for prog in (*_packet_programs(), _disjoint(23), *(_steps_by_hand(k)[0] for k in ("upper half", "whole"))):
        for form in (prog, PG.packetize(prog)) if int(prog.steps["out_rank"].max()) <= 6 else (prog,):
            before = form.steps.copy()
            tags = PG.count_tags(form)
            assert (form.steps == before).all()
            np.testing.assert_array_equal(tags, PG.count_widths(form).steps["pad"][:, 0])


@pytest.mark.gpu
def test_device_records_carry_the_widths():
    """The records of a counter on the device are count_widths' (lane masks apart), whatever
    form or widths they had before."""
    from tensorsat_amd.executor import BatchCounter

    for prog in (*_packet_programs(), _disjoint(23), _steps_by_hand("upper half")[0]):
        stale = PG.count_widths(prog)
        forms = [prog, stale]
        if int(prog.steps["out_rank"].max()) <= 6:
            forms.append(PG.packetize(prog))
        for form in forms:
            got = BatchCounter(form, widths=True).dp.steps.cpu().numpy().view(PG.STEP_DTYPE)
            want = PG.count_widths(form).steps
            tagged = want["pad"][:, 0] != 0
            if not tagged.any():  # counted by ts_batch_count, which ignores them
                continue
            np.testing.assert_array_equal(got["pad"][tagged], want["pad"][tagged])
            np.testing.assert_array_equal(got["flags"][tagged], want["flags"][tagged])
            assert not (got["flags"][~tagged] & PG.STEP_WIDTHS).any()
            for name in ("lhs_off", "rhs_off", "out_off", "out_rank", "sum_rank", "c_lpos", "o_rpos"):
                np.testing.assert_array_equal(got[name], want[name])


@pytest.mark.gpu
@pytest.mark.parametrize("widths", [True, False])
def test_both_kernels_count_alike(widths):
    """Edges of uint32 and uint64, brute force, wide and general steps, by either kernel."""
    from tensorsat_amd.executor import BatchCounter
    from wide_steps import wide_sum_program

    for m in (1, 9, 10, 11, 20, 21, 22):
        assert BatchCounter(_disjoint(m), widths=widths).run() == [7**m], m
    with pytest.raises(OverflowError):
        BatchCounter(_disjoint(23), widths=widths).run()
    for n, width in ((14, 3), (20, 9), (22, 12), (24, 16)):
        cnfs = [CNFInstance.random(3, n, int(r * n), rng=40 * n + i) for i, r in enumerate((1.0, 2.0, 3.0))]
        counter = BatchCounter(PG.sat_batch(cnfs, width=width), widths=widths)
        assert counter.widths is widths
        assert counter.run() == [brute.count(c.num_vars, c.clauses) for c in cnfs]
    for permute in (True, False):
        prog, _ = wide_sum_program(3, out_wires=(), n=10, density=0.5, permute=permute)
        assert BatchCounter(prog, widths=widths).run() == BatchCounter(prog, widths=not widths).run()


@pytest.mark.gpu
def test_widths_come_with_large_tensors():
    from tensorsat_amd.executor import BatchCounter

    for width in (8, 14):
        prog = PG.sat_batch([CNFInstance.random(3, 40, 120, rng=5)], width=width, max_cubes=4)
        assert BatchCounter(prog).widths is (int(prog.steps["out_rank"].max()) >= BatchCounter.WIDTHS_RANK)
