"""
GPU parity of gang execution (ts_program_run_gang): several jobs of one program advanced
together phase by phase.  Each job's result, read from its arena, equals the oracle's
byte for byte and its flag equals "the result has a nonzero entry", for gangs of cubes
with different step structures (cubes of twelve n=70 instances, more than two launches'
worth of jobs) and of slices with one structure (the n=40 greedy tree), across the small-step
threshold; decisions through gangs equal DPLL.
"""

import numpy as np
import pytest

from oracle import dpll
from oracle import executor as OX
from tensorsat_amd import program as PG
from tensorsat_amd.sat import CNFInstance
from tensorsat_amd.workloads import plain_cpu_3sat, single_3sat

pytestmark = pytest.mark.gpu


def _check_gang(prog, first, count, mode, small_bits, oracle_jobs):
    import torch

    from tensorsat_amd.executor import DeviceProgram, gang_stride, run_gang, run_job_fused

    dp = DeviceProgram(prog)
    stride = gang_stride(dp)
    arena = torch.full((count * stride,), 5, dtype=torch.uint8, device="cuda")
    flags = run_gang(dp, first, count, mode, arena=arena, small_bits=small_bits).cpu().numpy()
    torch.cuda.synchronize()
    jobs = prog.jobs
    for g in range(count):
        j = first + g
        r0, rr = int(jobs["result_off"][j]), int(jobs["result_rank"][j])
        got = arena[g * stride + r0 : g * stride + r0 + (1 << rr)].cpu().numpy()
        one = run_job_fused(dp, j, mode, small_bits=12).cpu().numpy()
        np.testing.assert_array_equal(got, one, err_msg=f"job {j}: gang vs one job at a time")
        assert flags[g] == int(got.any()), f"job {j} flag"
        if j in oracle_jobs:
            ref, _ = OX.run_job(prog, j, mode)
            np.testing.assert_array_equal(got, ref.reshape(-1), err_msg=f"job {j}: gang vs oracle")


@pytest.mark.parametrize("small_bits", [12, 6, 0])
@pytest.mark.parametrize("mode", ["GT0", "MOD256"])
def test_gang_of_cubes_with_different_structures(mode, small_bits):
    cnfs = [CNFInstance.random(3, 70, 290, rng=900 + i) for i in range(12)]
    prog = PG.sat_batch(cnfs, width=14, plan_trials=1)
    n = len(prog.jobs)
    print(f"cubes {n} mode {mode} small_bits {small_bits}", flush=True)
    assert n > 128 and np.unique(prog.jobs["num_steps"]).size > 10  # three launches' worth, mixed shapes
    _check_gang(prog, 0, n, mode, small_bits, oracle_jobs={0, 1, 63, 64, 128, n - 1})


@pytest.mark.parametrize("mode", ["GT0", "MOD256"])
def test_gang_of_slices_with_one_structure(mode):
    from tensorsat_amd.contractions import PlannedContraction
    from tensorsat_amd.rel import DeviceRel

    cnf = plain_cpu_3sat(0)
    d = (cnf.inputs(None) >> cnf.diagram()).flatten()
    c = PlannedContraction(DeviceRel, d.wiring, optimize="greedy", slicing_target=22)
    prog = c.contract_program(d)
    print(f"slices {len(prog.jobs)} sliced wires {len(c.tree.sliced)}", flush=True)
    _check_gang(prog, 3, 70, mode, 12, oracle_jobs={3, 40, 72})


@pytest.mark.parametrize("gang,lookahead", [(0, False), (4, True), (32, False), (64, True)])
def test_gang_decisions_match_dpll(gang, lookahead):
    from tensorsat_amd.single import decide

    for seed in range(3):
        cnf = single_3sat(seed)
        r = decide(cnf, width=22, gang=gang, first_gang=min(8, gang) if gang else 8, lookahead=lookahead)
        print(f"seed {seed} gang {gang}: verdict {r.value} cubes {r.cubes_run}/{r.cubes}", flush=True)
        assert r.value == int(dpll.solve(cnf.num_vars, cnf.clauses))
        assert r.cubes_run <= r.stats["cubes_launched"] <= r.cubes


def test_gang_rejects_bad_arguments():
    import torch

    from tensorsat_amd.executor import DeviceProgram, run_gang

    prog = PG.sat_batch([single_3sat(0)], width=12, max_cubes=4, plan_trials=1)
    dp = DeviceProgram(prog)
    with pytest.raises(ValueError):
        run_gang(dp, 2, 10)
    with pytest.raises(ValueError):
        run_gang(dp, 0, 2, arena=torch.empty(16, dtype=torch.uint8, device="cuda"))


@pytest.mark.parametrize("seed,k", [(0, 10), (1, 5)])
def test_gang_packed_rows(seed, k):
    """n=40 slices whose largest steps have 2^k-byte rows (k = 10 and 5) read by many
    outputs: gang execution packs those rows into bit masks first; every result equals
    the unpacked single-job path, in both epilogues."""
    from tensorsat_amd.contractions import PlannedContraction
    from tensorsat_amd.executor import DeviceProgram, gang_stride, run_gang, run_job_fused
    from tensorsat_amd.rel import DeviceRel

    import torch

    cnf = plain_cpu_3sat(seed)
    d = (cnf.inputs(None) >> cnf.diagram()).flatten()
    prog = PlannedContraction(DeviceRel, d.wiring, optimize="greedy", slicing_target=26).contract_program(d)
    st = prog.steps[: int(prog.jobs["num_steps"][0])]
    assert np.any((st["sum_rank"] == k) & (st["out_rank"] >= 12) & ((st["flags"] & 1) != 0))
    dp = DeviceProgram(prog)
    stride = gang_stride(dp)
    assert stride > int(prog.jobs["arena_elems"].max()) + 255  # room for the masks
    for mode in ("GT0", "MOD256"):
        arena = torch.empty(4 * stride, dtype=torch.uint8, device="cuda")
        flags = run_gang(dp, 0, 4, mode, arena=arena).cpu().numpy()
        for g in range(4):
            r0, rr = int(prog.jobs["result_off"][g]), int(prog.jobs["result_rank"][g])
            got = arena[g * stride + r0 : g * stride + r0 + (1 << rr)].cpu().numpy()
            want = run_job_fused(dp, g, mode).cpu().numpy()
            np.testing.assert_array_equal(got, want, err_msg=f"slice {g} {mode}")
            assert flags[g] == int(want.any())


def _first_packed_step(prog, j):
    """Index in job j of its first step whose rows gang execution packs, or None."""
    b, n = int(prog.jobs["step_begin"][j]), int(prog.jobs["num_steps"][j])
    for i, st in enumerate(prog.steps[b : b + n]):
        ro, k = int(st["out_rank"]), int(st["sum_rank"])
        held = (st["o_lpos"][:ro] != PG.NOPOS) != (st["o_rpos"][:ro] != PG.NOPOS)
        if (st["flags"] & 3) == PG.STEP_KINNER and 4 <= k <= 5 and ro >= 12 and held.sum() >= 2:
            return i
    return None


def test_gang_packed_rows_of_different_jobs():
    """Jobs of different arena sizes whose packed steps run in one launch: each job's masks are
    its own.  The gang runs every job up to its first packed step, whose whole output is
    compared with the one-step-at-a-time runner's."""
    import torch

    from tensorsat_amd.executor import DeviceProgram, gang_stride, run_gang, run_job

    progs, rng = [], np.random.default_rng(4)
    while len(progs) < 6:
        cnf = CNFInstance.random(3, 110, 440, rng=int(rng.integers(1 << 30)))
        p = PG.sat_batch([cnf], width=24, max_cubes=1)
        if len(p.jobs) == 1 and _first_packed_step(p, 0) is not None:
            progs.append(p)
    prog = PG.concat(progs, [np.array([i]) for i in range(6)], 6)
    assert len(set(prog.jobs["arena_elems"].tolist())) > 1
    dp = DeviceProgram(prog)
    stride = gang_stride(dp)
    last = [_first_packed_step(prog, j) for j in range(6)]
    want = [run_job(dp, j, "GT0", keep_intermediates=True)[1][last[j]] for j in range(6)]
    for j in range(6):
        dp.jobs_host["num_steps"][j] = last[j] + 1
        dp.jobs_host["result_off"][j] = prog.steps["out_off"][prog.jobs["step_begin"][j] + last[j]]
        dp.jobs_host["result_rank"][j] = prog.steps["out_rank"][prog.jobs["step_begin"][j] + last[j]]
    for mode in ("GT0", "MOD256"):
        for small_bits in (12, 0):
            arena = torch.full((6 * stride,), 255, dtype=torch.uint8, device="cuda")
            run_gang(dp, 0, 6, mode, arena=arena, small_bits=small_bits)
            for j in range(6):
                o, n = j * stride + int(dp.jobs_host["result_off"][j]), 1 << int(dp.jobs_host["result_rank"][j])
                print(f"{mode} small {small_bits} job {j}: step {last[j]}, {n} outputs", flush=True)
                assert torch.equal(arena[o : o + n], want[j])


def _dense_program(rng, shapes):
    """One job per (m, n, b, k) in ``shapes``: a single dense record over random leaves, all
    records of a shape alike."""
    steps, jobs, leaves, layouts = [], [], [], {}
    for i, (m, n, b, k) in enumerate(shapes):
        ro = m + n + b
        side = layouts.setdefault((m, n, b, k), rng.permutation(np.repeat([0, 1, 2], [m, n, b])))
        st, rec = np.zeros(1, PG.STEP_DTYPE), np.zeros(1, PG.JOB_DTYPE)
        for name, other in (("o_lpos", 1), ("o_rpos", 0)):
            st[name] = PG.NOPOS
            st[name][0, :ro][side != other] = k + np.arange((side != other).sum())
        for name in ("c_lpos", "c_rpos"):
            st[name] = PG.NOPOS
            st[name][0, :k] = range(k)
        lsz, rsz = 1 << (k + m + b), 1 << (k + n + b)
        st["lhs_rank"], st["rhs_rank"], st["out_rank"], st["sum_rank"] = k + m + b, k + n + b, ro, k
        st["rhs_off"], st["out_off"], st["flags"] = lsz, lsz + rsz, PG.STEP_KINNER
        rec["step_begin"], rec["num_steps"], rec["instance"] = i, 1, i
        rec["leaf_begin"], rec["num_leaf_bytes"] = sum(x.size for x in leaves), lsz + rsz
        rec["result_off"], rec["result_rank"], rec["max_rank"] = lsz + rsz, ro, max(ro, k + b + max(m, n))
        rec["arena_elems"] = lsz + rsz + (1 << ro)
        steps.append(st)
        jobs.append(rec)
        leaves.append((rng.random(lsz + rsz) < rng.choice([0.02, 0.1, 1.0])).astype(np.uint8))
    prog = PG.Program(np.concatenate(jobs), np.concatenate(steps), np.concatenate(leaves),
                      np.zeros((len(shapes), PG.NSTAT), np.int64), {})
    PG.validate(prog)
    return prog


@pytest.mark.parametrize("mode", ["GT0", "MOD256"])
def test_gang_of_dense_steps(mode):
    """Matrix-core steps of several jobs in one launch: more jobs than one launch holds, changes
    of shape, two shapes in turn, and jobs without such a step between them."""
    import torch

    from tensorsat_amd.executor import DeviceProgram, gang_stride, run_gang, run_job

    a, b, c = (5, 4, 1, 8), (4, 6, 0, 6), (6, 5, 2, 9)
    slow = (2, 3, 4, 6)  # too few bits on either side
    shapes = [a] * 67 + [b] * 3 + [c, a, c, a, a] + [slow, b, slow, slow, b, c, c]
    prog = _dense_program(np.random.default_rng(12), shapes)
    dp = DeviceProgram(prog)
    stride, n = gang_stride(dp), len(shapes)
    arena = torch.full((n * stride,), 255, dtype=torch.uint8, device="cuda")
    flags = run_gang(dp, 0, n, mode, arena=arena, small_bits=0).cpu().numpy()
    seen = set()
    for j in range(n):
        print(f"{mode} job {j} shape {shapes[j]}", flush=True)
        want = OX.run_job(prog, j, mode)[0].reshape(-1)
        at = j * stride + int(prog.jobs["result_off"][j])
        np.testing.assert_array_equal(arena[at : at + want.size].cpu().numpy(), want)
        np.testing.assert_array_equal(run_job(dp, j, mode)[0].cpu().numpy().reshape(-1), want)
        assert flags[j] == int(want.any())
        seen.add(want.tobytes())
    assert len(seen) > n // 2  # the jobs' results differ


@pytest.mark.parametrize("mode", ["GT0", "MOD256"])
def test_staged_runs_at_the_limit(mode):
    """Runs of small steps whose tensors end at the last entry that is staged in LDS (65536), one
    piece below and one above, beside jobs that end far below."""
    import torch

    from tensorsat_amd.executor import DeviceProgram, gang_stride, run_gang

    parts, want = [], []
    for i, end in enumerate((65536, None, 65520, 65552, None, 65536)):
        w = CNFInstance.random(3, 10, 35, rng=60 + i)
        d = (w.inputs("_" * 10) >> w.diagram()).flatten()
        p = PG.compile_network(d.wiring, list(d.blocks), PG.elim(d.wiring, trials=1))
        assert len(p.steps) >= 65
        shift = 0 if end is None else end - int(p.jobs["arena_elems"][0])
        for name in ("lhs_off", "rhs_off", "out_off"):
            p.steps[name] += shift
        for name in ("num_leaf_bytes", "result_off", "arena_elems"):
            p.jobs[name] += shift
        top = max(int(p.steps["out_off"][k]) + (1 << int(p.steps["out_rank"][k])) for k in range(len(p.steps)))
        p.leaves = np.concatenate([np.full(shift, 3, np.uint8), p.leaves])
        assert end is None or top == end
        parts.append(p)
        want.append(OX.run_job(p, 0, mode)[0].reshape(-1))
    prog = PG.concat(parts, [np.array([i]) for i in range(6)], 6)
    PG.validate(prog)
    dp = DeviceProgram(prog)
    stride = gang_stride(dp)
    for small_bits in (12, 9):
        arena = torch.full((6 * stride,), 255, dtype=torch.uint8, device="cuda")
        flags = run_gang(dp, 0, 6, mode, arena=arena, small_bits=small_bits).cpu().numpy()
        for j in range(6):
            at = j * stride + int(prog.jobs["result_off"][j])
            print(f"{mode} small {small_bits} job {j}", flush=True)
            np.testing.assert_array_equal(arena[at : at + want[j].size].cpu().numpy(), want[j])
            assert flags[j] == int(want[j].any())
