"""
Performance cases: the work a program gives this framework, through its public entry
points, with inputs made from a seed.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare(case, seed)`` makes what a program holds before the call, ``run(state)`` is one
pass, ``work(case)`` the bytes and operations a pass cannot do without, ``tolerance(case)``
how far two correct implementations may differ, and ``exact(case, seed)`` the result in
64-bit arithmetic where the outputs are computed numbers.

Verdicts, counts and relations are whole numbers: every correct implementation gives the
same ones.  Only the learned planner's network computes floating-point outputs.
"""

import math

import numpy as np
import torch

from tensorsat_amd.contractions import PlannedContraction
from tensorsat_amd.executor import BatchCounter, DeviceProgram, gang_stride, run_gang
from tensorsat_amd.learn import data as learn_data
from tensorsat_amd.learn import graph as learn_graph
from tensorsat_amd.learn.model import GNN, HID, LAYERS
from tensorsat_amd.learn.propose import WEIGHTS
from tensorsat_amd.program import concat, sat_batch
from tensorsat_amd.rel import DeviceRel
from tensorsat_amd.sat import CNFInstance
from tensorsat_amd.search import SearchSolver


def listed():
    return [
        # The reference's call shape on a small network: the relation of all solutions of a
        # 10-variable 3-SAT instance, contracted pairwise along a planned tree.  The
        # smallest calls: about a hundred contractions of a few bytes each.
        {"name": "relation_n10", "kind": "relation", "vars": 10, "ratio": 3.5, "mode": "GT0"},
        # A request of a few dozen instances, from CNF objects to verdicts on the host:
        # packing, upload, one search launch, read-back.
        {"name": "decide_64", "kind": "decide_host", "instances": 64, "lo": 20, "hi": 60, "width": 6, "split": 8.0},
        # The headline workload: 4096 uneven random 3-SAT instances (n in 20..80, ratio 4.26
        # and 3.5), packed clauses resident, one decision of the whole batch.
        {"name": "decide_4096", "kind": "decide", "instances": 4096, "lo": 20, "hi": 80, "width": 6, "split": 8.0},
        # Exact model counts of a few instances by the exhaustive device search.
        {"name": "count_search_8", "kind": "count_search", "instances": 8, "lo": 50, "hi": 60, "split_bits": 10},
        # Exact model count of one n=100, m=300 instance over its cubes (64-bit counts).
        {"name": "count_n100", "kind": "count", "vars": 100, "ratio": 3.0, "width": 18},
        # Large decisions (n=120): a gang of the first cubes of a few instances, with tensors
        # of up to 2^26 entries.
        {"name": "cubes_n120", "kind": "cubes", "vars": 120, "ratio": 4.0, "width": 26, "instances": 8, "each": 1,
         "gang": 8, "mode": "GT0"},
        # The same for the reference's own kind of tree: slices of a greedy tree (n=40) cut to
        # 2^26 entries, a gang of slices with identical steps.
        {"name": "slices_n40", "kind": "slices", "vars": 40, "ratio": 3.5, "target": 26, "gang": 16, "mode": "GT0"},
        # Composition of two binary relations over 8192 elements: a dense Boolean product.
        {"name": "compose_8192", "kind": "compose", "rows": 8192, "inner": 8192, "cols": 8192, "mode": "GT0"},
        # One large pairwise contraction as a tree walk issues it: many wires, one summed,
        # the operands' wires in unrelated orders.
        {"name": "contract_26", "kind": "contract", "lhs": 25, "rhs": 24, "shared": 22, "summed": 1, "layout": 3,
         "mode": "GT0"},
        # Port algebra on the largest relation: a permutation of all 27 bit ports, and an
        # existential reduction to 16 of them.
        {"name": "permute_27", "kind": "rewire", "rank": 27, "keep": 27, "layout": 5, "mode": "GT0"},
        {"name": "reduce_27", "kind": "rewire", "rank": 27, "keep": 16, "layout": 6, "mode": "GT0"},
        # A training step's forward and backward pass of the learned planner's network on a
        # batch of 32 generated k-SAT instances (about 90 000 clauses).
        {"name": "gnn_train_32", "kind": "gnn", "instances": 32, "train": True},
    ]


def _log_int(rng, lo, hi):
    """An integer in lo..hi, uniform over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["relation", "decide_host", "decide", "count_search", "count", "cubes", "slices", "compose",
                       "contract", "rewire", "gnn"])
    mode = rng.choice(["GT0", "GT0", "MOD256"])
    if kind == "relation":
        return {"kind": kind, "vars": rng.randint(6, 12), "ratio": round(rng.uniform(2.0, 3.5), 3), "mode": mode}
    if kind in ("decide_host", "decide"):
        lo = rng.randint(20, 50)
        return {"kind": kind, "instances": _log_int(rng, 24, 512) if kind == "decide_host" else _log_int(rng, 64, 4096),
                "lo": lo, "hi": rng.randint(lo, 80), "width": rng.choice([4, 6]), "split": rng.choice([8.0, 32.0])}
    if kind == "count_search":
        lo = rng.randint(30, 50)
        return {"kind": kind, "instances": rng.randint(2, 12), "lo": lo, "hi": rng.randint(lo, 58),
                "split_bits": rng.randint(6, 10)}
    if kind == "count":
        return {"kind": kind, "vars": rng.randint(60, 92), "ratio": round(rng.uniform(3.0, 3.4), 3),
                "width": rng.randint(16, 18)}
    if kind == "cubes":
        num, each = rng.choice([(4, 2), (5, 2), (6, 1), (7, 1), (8, 1), (9, 1)])
        return {"kind": kind, "vars": rng.randint(100, 120), "ratio": round(rng.uniform(3.9, 4.05), 3),
                "width": rng.randint(20, 26), "instances": num, "each": each, "gang": num * each, "mode": mode}
    if kind == "slices":
        return {"kind": kind, "vars": rng.randint(38, 40), "ratio": round(rng.uniform(3.3, 3.6), 3),
                "target": rng.randint(24, 26), "gang": rng.randint(5, 16), "mode": mode}
    if kind == "compose":
        return {"kind": kind, "rows": _log_int(rng, 60, 8192), "inner": _log_int(rng, 60, 8192),
                "cols": _log_int(rng, 60, 8192), "mode": mode}
    if kind == "contract":
        summed = rng.randint(0, 4)
        shared = rng.randint(summed, 20)
        out = rng.randint(16, 26)  # lhs-only + rhs-only + shared - summed out wires
        own = max(0, out - (shared - summed))
        left = rng.randint(0, own)
        return {"kind": kind, "lhs": min(26, shared + left), "rhs": min(26, shared + own - left), "shared": shared,
                "summed": summed, "layout": rng.randint(0, 10**6), "mode": mode}
    if kind == "rewire":
        rank = rng.randint(14, 27)
        return {"kind": kind, "rank": rank, "keep": rank if rng.random() < 0.4 else rng.randint(2, rank - 1),
                "layout": rng.randint(0, 10**6), "mode": mode}
    return {"kind": kind, "instances": _log_int(rng, 6, 32), "train": rng.random() < 0.5}


# ---- inputs -------------------------------------------------------------------------


def _clauses(rng, n, m, k=3):
    """m random clauses of k distinct variables out of n, signs at random."""
    v = rng.integers(1, n + 1, size=(m, k))
    while True:
        s = np.sort(v, axis=1)
        bad = (s[:, 1:] == s[:, :-1]).any(axis=1)
        if not bad.any():
            break
        v[bad] = rng.integers(1, n + 1, size=(int(bad.sum()), k))
    return np.where(rng.integers(0, 2, size=(m, k)) == 0, v, -v)


def _cnf(rng, n, ratio):
    return CNFInstance(n, _clauses(rng, n, int(round(ratio * n))).tolist())


def _batch(case, seed, ratios):
    rng = np.random.default_rng(seed)
    return [_cnf(rng, int(rng.integers(case["lo"], case["hi"] + 1)), ratios[i % len(ratios)])
            for i in range(case["instances"])]


def _relation(shape, seed, density=0.5):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = torch.rand(math.prod(shape), device="cuda", generator=g) < density
    return DeviceRel.from_numpy(t.to(torch.uint8).cpu().numpy().reshape(shape))


def _contract_wires(case):
    """lhs, rhs and out wires: out in lhs order, then the rhs-only wires, as a tree walk
    writes them; everything else in random order."""
    rng = np.random.default_rng(case["layout"])
    shared = list(range(case["shared"]))
    lhs = shared + list(range(100, 100 + case["lhs"] - case["shared"]))
    rhs = shared + list(range(200, 200 + case["rhs"] - case["shared"]))
    lhs, rhs = ([int(w) for w in rng.permutation(ws)] for ws in (lhs, rhs))
    gone = {int(w) for w in rng.permutation(shared)[: case["summed"]]} if shared else set()
    out = [w for w in lhs if w not in gone] + [w for w in rhs if w not in gone and w not in lhs]
    return lhs, rhs, out


def _ports(case):
    rng = np.random.default_rng(case["layout"])
    if case["keep"] == case["rank"]:
        return [int(p) for p in rng.permutation(case["rank"])]
    return sorted(int(p) for p in rng.choice(case["rank"], size=case["keep"], replace=False))


def _program(case, seed):
    """The compiled program of a "count", "cubes" or "slices" case: instances that leave no
    cube, or fewer cubes or slices than the case takes, are passed over for the next."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "cubes":
        progs = []
        while len(progs) < case["instances"]:
            p = sat_batch([_cnf(rng, case["vars"], case["ratio"])], width=case["width"], max_cubes=case["each"])
            if len(p.jobs) == case["each"]:
                progs.append(p)
        return concat(progs, [np.array([i]) for i in range(len(progs))], len(progs))
    while True:
        cnf = _cnf(rng, case["vars"], case["ratio"])
        if case["kind"] == "slices":
            d = (cnf.inputs(None) >> cnf.diagram()).flatten()
            c = PlannedContraction(DeviceRel, d.wiring, optimize="greedy", slicing_target=case["target"])
            prog = c.contract_program(d)
        else:
            prog = sat_batch([cnf], width=case["width"], plan_trials=1)
        if len(prog.jobs) >= case.get("gang", 1):
            return prog


def _graph(case, seed):
    """k in {3, 4, 5}, n from 150 to 300 evenly over the batch, so that every seed's batch
    has the same size."""
    num = case["instances"]
    return learn_graph.build([learn_data.ksat(seed * 1000 + i, k=3 + i % 3, n=150 + 150 * i // max(1, num - 1))
                              for i in range(num)])


def _target(g, seed):
    return np.random.default_rng(seed).random(g.num_vars).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "relation":
        cnf = _cnf(np.random.default_rng(seed), case["vars"], case["ratio"])
        d = (cnf.inputs("_" * case["vars"]) >> cnf.diagram()).flatten()
        return {"case": case, "diagram": d, "contraction": PlannedContraction(DeviceRel, d.wiring)}
    if kind == "decide_host":
        cnfs = _batch(case, seed, (4.26, 3.5))
        return {"case": case, "cnfs": cnfs, "solver": SearchSolver(width=case["width"], split_target=case["split"])}
    if kind == "decide":
        solver = SearchSolver(width=case["width"], split_target=case["split"])
        solver.prepare(_batch(case, seed, (4.26, 3.5)))
        return {"case": case, "solver": solver}
    if kind == "count_search":
        solver = SearchSolver(width=6, split_target=1e-9, max_split=case["split_bits"], budget=4096, count=True,
                              max_nodes=1 << 40)
        solver.prepare(_batch(case, seed, (3.0,)))
        return {"case": case, "solver": solver}
    if kind == "count":
        return {"case": case, "counter": BatchCounter(_program(case, seed))}
    if kind in ("cubes", "slices"):
        dp = DeviceProgram(_program(case, seed))
        return {"case": case, "dp": dp,
                "arena": torch.empty(case["gang"] * gang_stride(dp), dtype=torch.uint8, device="cuda")}
    if kind == "compose":
        p = case["inner"] ** -0.5  # both values frequent in the result
        return {"case": case, "lhs": _relation((case["rows"], case["inner"]), 2 * seed, p),
                "rhs": _relation((case["inner"], case["cols"]), 2 * seed + 1, p)}
    if kind == "contract":
        return {"case": case, "lhs": _relation((2,) * case["lhs"], 2 * seed),
                "rhs": _relation((2,) * case["rhs"], 2 * seed + 1), "wires": _contract_wires(case)}
    if kind == "rewire":
        # sparse enough that a reduction leaves both values
        p = 0.5 if case["keep"] == case["rank"] else min(0.5, 2.0 ** (case["keep"] - case["rank"]))
        return {"case": case, "box": _relation((2,) * case["rank"], seed, p), "ports": _ports(case)}
    g = _graph(case, seed)
    # Training starts from a fresh network, scoring uses the shipped weights.
    return {"case": case, "model": GNN(seed=0) if case["train"] else GNN.load(WEIGHTS),
            "graph": learn_graph.DeviceGraph(g), "target": torch.from_numpy(_target(g, seed)).cuda()}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "relation":
        with DeviceRel.mode_scope(case["mode"]):
            box = state["contraction"].contract(state["diagram"])
        return box.data[: 1 << box.device_bits]
    if kind == "decide_host":
        return state["solver"].run(state["cnfs"])
    if kind == "decide":
        state["solver"].launch()
        return state["solver"].d_verdicts
    if kind == "count_search":
        state["solver"].launch()
        return np.array(state["solver"].counts(), dtype=np.int64)
    if kind == "count":
        return state["counter"].run()
    if kind in ("cubes", "slices"):
        return run_gang(state["dp"], 0, case["gang"], case["mode"], arena=state["arena"])
    with DeviceRel.mode_scope(case.get("mode", "GT0")):
        if kind == "compose":
            box = DeviceRel.contract2(state["lhs"], [0, 1], state["rhs"], [1, 2], [0, 2])
            return box.data[: 1 << box.device_bits]
        if kind == "contract":
            lhs, rhs, out = state["wires"]
            box = DeviceRel.contract2(state["lhs"], lhs, state["rhs"], rhs, out)
            return box.data[: 1 << box.device_bits]
        if kind == "rewire":
            box = state["box"].rewire(state["ports"])
            return box.data[: 1 << box.device_bits]
    model = state["model"]
    if not case["train"]:
        return model.forward(state["graph"])[0]
    y, loss = model.forward(state["graph"], target=state["target"], train=True)
    return {"y": y, "loss": loss, "grad": model.g}


# ---- what a pass cannot do without -----------------------------------------------------


def _steps_work(case):
    """Leaves and step records read once, the AND and the sum of every step's terms, for
    the program of seed 0."""
    prog = _program(case, 0)
    jobs = prog.jobs if case["kind"] == "count" else prog.jobs[: case["gang"]]
    steps = np.concatenate([prog.steps[b : b + n] for b, n in zip(jobs["step_begin"], jobs["num_steps"])])
    terms = 2.0 ** (steps["out_rank"].astype(np.float64) + steps["sum_rank"])
    return {"bytes": float(jobs["num_leaf_bytes"].sum()) + 128.0 * len(steps), "flops": 2.0 * float(terms.sum())}


def work(case):
    kind = case["kind"]
    if kind == "relation":
        m = int(round(case["ratio"] * case["vars"]))
        return {"bytes": 8.0 * m + 2.0 ** case["vars"], "flops": 2.0 * m * 2.0 ** case["vars"]}
    if kind in ("decide_host", "decide", "count_search"):
        clauses = case["instances"] * (case["lo"] + case["hi"]) / 2 * (3.0 if kind == "count_search" else 3.88)
        return {"bytes": 4.0 * clauses + 20.0 * case["instances"], "flops": 0.0}
    if kind in ("count", "cubes", "slices"):
        return _steps_work(case)
    if kind == "compose":
        r, i, c = case["rows"], case["inner"], case["cols"]
        return {"bytes": float(r * i + i * c + r * c), "flops": 2.0 * r * i * c}
    if kind == "contract":
        lhs, rhs, out = _contract_wires(case)
        return {"bytes": 2.0 ** len(lhs) + 2.0 ** len(rhs) + 2.0 ** len(out),
                "flops": 2.0 * 2.0 ** (len(out) + case["summed"])}
    if kind == "rewire":
        return {"bytes": 2.0 ** case["rank"] + 2.0 ** case["keep"], "flops": 2.0 ** case["rank"]}
    g = _graph(case, 0)
    v, c, e, h = g.num_vars, g.num_clauses, len(g.c2v_col), HID
    flops = 2.0 * (v + c) * h * (learn_graph.FEAT + LAYERS * 3 * h) + LAYERS * 4.0 * e * h
    weights = 2 * learn_graph.FEAT * h + LAYERS * 6 * h * h
    nbytes = 2.0 * learn_graph.FEAT * (v + c) + 16.0 * e + 2.0 * weights + 4.0 * v
    if case["train"]:
        flops, nbytes = 3 * flops, nbytes + 4.0 * weights + 4.0 * v
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Scores and gradients of a 13-layer network that keeps its activations in bf16 (sums in
    # fp32): against 64 bits the scores are off by 0.0025 and the gradients by 0.002 to 0.006.
    return {"rel": 0.02, "max": 0.5} if case["kind"] == "gnn" else "exact"


def _signed_sums(rowptr, col, weight, rows, x):
    """Sums over the positive and over the negative incidences of every row, weighted."""
    row = torch.repeat_interleave(torch.arange(rows, device=x.device), rowptr[1:].long() - rowptr[:-1].long())
    out = []
    for part in (weight > 0, weight < 0):
        z = torch.zeros(rows, x.shape[1], dtype=x.dtype, device=x.device)
        out.append(z.index_add(0, row[part], weight[part].abs().to(x.dtype)[:, None] * x[col[part].long()]))
    return out


def exact(case, seed):
    if case["kind"] != "gnn":
        return None  # verdicts, counts and relations: whole numbers, compared as they are
    state = prepare(case, seed)
    model, dg = state["model"], state["graph"]
    # The weights and features as the network holds them for its products (bf16), biases and
    # head in fp32; everything after that in 64 bits.
    p = {}
    for name, (off, shape) in model.layout.items():
        src = model.pbf if name.startswith("W") else model.p
        p[name] = src[off : off + math.prod(shape)].double().reshape(shape).requires_grad_(case["train"])
    c2v = (dg.c2v_rowptr, dg.c2v_col, dg.c2v_w, dg.C)
    v2c = (dg.v2c_rowptr, dg.v2c_col, dg.v2c_w, dg.V)
    hv = torch.relu(dg.var_feat.double() @ p["W_vin"] + p["b_vin"])
    hc = torch.relu(dg.clause_feat.double() @ p["W_cin"] + p["b_cin"])
    for k in range(LAYERS):
        hc = torch.relu(torch.cat([hc, *_signed_sums(*c2v, hv)], 1) @ p[f"Wc{k}"] + p[f"bc{k}"])
        hv = torch.relu(torch.cat([hv, *_signed_sums(*v2c, hc)], 1) @ p[f"Wv{k}"] + p[f"bv{k}"])
    y = hv @ p["w_out"] + p["b_out"]
    if not case["train"]:
        return y.detach()
    loss = (y - state["target"].double()).square().mean()
    loss.backward()
    grad = torch.cat([p[name].grad.reshape(-1) for name in model.layout])
    return {"y": y.detach(), "loss": loss.detach().reshape(1), "grad": grad}
