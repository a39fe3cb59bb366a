"""
Steps of short rows (0..3 summed bits, innermost) whose two, one or none of the lowest out bits
sit in order right above them in each operand: single records against the oracle, exact, one
step at a time and through a gang launch.
"""

import numpy as np
import pytest

from oracle import executor as OX
from tensorsat_amd import program as PG

pytestmark = pytest.mark.gpu


def _positions(rng, held, nc, in_order):
    """Positions of the held out bits above nc summed ones: the held ones among the first
    ``in_order`` out bits in place, the others shuffled so that no more are."""
    first = [j for j in held if j < in_order]
    rest = [j for j in held if j >= in_order]
    while True:
        order = first + [rest[int(i)] for i in rng.permutation(len(rest))]
        if in_order == 2 or in_order not in held or len(rest) < 2 or order[len(first)] != in_order:
            return {j: nc + i for i, j in enumerate(order)}


def _program(rng, jobs, ro, nc, in_order, unary):
    """``jobs`` jobs of one record each, all of one shape."""
    steps, leaves, recs = [], [], []
    for _ in range(jobs):
        st = np.zeros(1, PG.STEP_DTYPE)
        for name in ("o_lpos", "o_rpos", "c_lpos", "c_rpos"):
            st[name] = PG.NOPOS
        bits = np.arange(ro)
        left = bits if unary else bits[rng.random(ro) < 0.7]
        right = np.zeros(0, int) if unary else np.union1d(np.setdiff1d(bits, left), bits[rng.random(ro) < 0.6])
        off = 0
        for pos, cpos, name, held in (("o_lpos", "c_lpos", "lhs", left), ("o_rpos", "c_rpos", "rhs", right)):
            if name == "rhs" and unary:
                st["rhs_off"] = st["lhs_off"]
                continue
            for j, p in _positions(rng, [int(b) for b in held], nc, in_order).items():
                st[pos][0, j] = p
            st[cpos][0, :nc] = range(nc)
            st[f"{name}_off"], st[f"{name}_rank"] = off, nc + len(held)
            off += max(16, 1 << (nc + len(held)))
        st["out_off"], st["out_rank"], st["sum_rank"] = off, ro, nc
        st["flags"] = PG.STEP_KINNER | (PG.STEP_NORHS if unary else 0)
        rec = np.zeros(1, PG.JOB_DTYPE)
        rec["step_begin"], rec["num_steps"] = len(steps), 1
        rec["leaf_begin"], rec["num_leaf_bytes"] = sum(x.size for x in leaves), off
        rec["result_off"], rec["result_rank"] = off, ro
        rec["arena_elems"], rec["max_rank"] = off + max(16, 1 << ro), max(ro, *(int(st[f"{x}_rank"][0]) for x in ("lhs", "rhs")))
        steps.append(st)
        recs.append(rec)
        leaves.append((rng.random(off) < 0.6 / (1 + nc / 2)).astype(np.uint8))
    prog = PG.Program(np.concatenate(recs), np.concatenate(steps), np.concatenate(leaves),
                      np.zeros((1, PG.NSTAT), np.int64), {})
    PG.validate(prog)
    return prog


@pytest.mark.parametrize("unary", [False, True])
@pytest.mark.parametrize("in_order", [0, 1, 2])
@pytest.mark.parametrize("nc", [0, 1, 2, 3])
def test_single_steps(nc, in_order, unary):
    import torch

    from tensorsat_amd.executor import DeviceProgram, gang_stride, run_gang, run_job

    rng = np.random.default_rng([nc, in_order, unary])
    for ro in (3, 4, 5, 8, 9, 12, 13, 17):
        prog = _program(rng, 6, ro, nc, in_order, unary)
        dp = DeviceProgram(prog)
        stride = gang_stride(dp)
        arena = torch.full((6 * stride,), 255, dtype=torch.uint8, device="cuda")
        for mode in ("GT0", "MOD256"):
            print(f"{ro} out bits, {nc} summed, {in_order} in order, unary {unary}, {mode}", flush=True)
            run_gang(dp, 0, 6, mode, arena=arena, small_bits=0)
            for j in range(6):
                want = OX.run_job(prog, j, mode)[0].reshape(-1)
                np.testing.assert_array_equal(run_job(dp, j, mode)[0].cpu().numpy().reshape(-1), want)
                at = j * stride + int(prog.jobs["result_off"][j])
                got = arena[at : (j + 1) * stride].cpu().numpy()
                np.testing.assert_array_equal(got[: 1 << ro], want)
                assert (got[max(16, 1 << ro) :] == 255).all()  # nothing past the output
