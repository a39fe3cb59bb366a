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
