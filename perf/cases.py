"""Performance cases: the work a user of this package has it do, through its public entry points.

A case is a dict of plain values.  ``prepare`` makes what a program holds before the call (a seeded graph
uploaded to an ``Executor``, a plan, a cost model); ``run`` is one call, as a program makes it.

Kinds
  match     ``Executor.run_gm``: one pattern counted over a resident graph (the ``run`` command line).
            k-clique presets take the local-bitmap passes, every other preset and every per-root
            count the reference's traversal order.
  batch     ``Executor.run_gm_batch``: many random patterns in one persistent launch.
  mce       ``Executor.run_mce``: maximal cliques of a degeneracy-ordered graph (the ``bk`` command line).
  view      ``Executor.transfer`` + ``run_gm`` of one view bin: what a pipeline consumer does per bin.
  schedule  ``Executor.learned_schedule``: features, cost model, order and parts of an uploaded view.
  train     ``Mlp.train``: the cost model fitted on logged roots.

Graphs: seeded R-MAT (.57, .19, .19, .05; drawn on the GPU, vertices permuted, isolated ones dropped),
Chung-Lu (power law 2.3) and the social family (Chung-Lu backbone plus planted communities).
"""
import importlib
import math

import numpy as np
import torch

g2 = importlib.import_module("g2-aimd_amd")
device = importlib.import_module("g2-aimd_amd.device")
batch = importlib.import_module("g2-aimd_amd.batch")

WAVES = 4096  # resident waves the learned schedule deals the roots over (16 per CU)


def listed():
    return [
        # a 4-clique count on a graph of a thousand vertices: launches and latency are all of it
        {"name": "k4-rmat10", "kind": "match", "graph": "rmat", "size": 10, "query": 24, "per_root": False},
        # triangles of an ordinary graph (174k vertices, 3.8M edges)
        {"name": "k3-rmat18", "kind": "match", "graph": "rmat", "size": 18, "query": 0, "per_root": False},
        # the headline: 4-cliques of R-MAT 22 (2.4M vertices, 64M edges)
        {"name": "k4-rmat22", "kind": "match", "graph": "rmat", "size": 22, "query": 24, "per_root": False},
        # a pattern that is no clique (4 vertices, 5 edges), with the count of every root
        {"name": "q2-chunglu100k-roots", "kind": "match", "graph": "chunglu", "size": 100000, "query": 2,
         "per_root": True},
        # a 5-vertex pattern with 8 edges on a small skewed graph (512 vertices, 6k edges)
        {"name": "q8-rmat9", "kind": "match", "graph": "rmat", "size": 9, "query": 8, "per_root": False},
        # a batch of random patterns of 3 to 5 vertices
        {"name": "batch48-rmat7", "kind": "batch", "graph": "rmat", "size": 7, "factor": 8, "queries": 48,
         "largest": 5},
        # the run that logs subtree sizes for training: a small skewed graph, per-root node counts
        {"name": "mce-rmat11-roots", "kind": "mce", "graph": "rmat", "size": 11, "per_root": True},
        # maximal cliques of the 100k-vertex Chung-Lu graph
        {"name": "mce-chunglu100k", "kind": "mce", "graph": "chunglu", "size": 100000, "per_root": False},
        # maximal cliques of a social graph (800k vertices, 22M edges)
        {"name": "mce-social800k", "kind": "mce", "graph": "social", "size": 800000, "per_root": False},
        # one of four view bins: upload, then the 4-cliques rooted in it
        {"name": "view-k4-rmat18", "kind": "view", "graph": "rmat", "size": 18, "query": 24, "bins": 4},
        # the learned schedule of a view
        {"name": "schedule-social200k", "kind": "schedule", "graph": "social", "size": 200000},
        # the cost model fitted on the logged roots of eight graphs
        {"name": "train-50k", "kind": "train", "rows": 50001, "epochs": 3, "batch": 512},
    ]


def log_size(rng, lo, hi):
    """an odd or even whole number, its logarithm uniform in [log lo, log hi]"""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("clique", "clique", "pattern", "pattern", "batch", "mce", "mce", "view", "schedule", "train"))
    if kind == "clique":
        query = rng.choice((0, 24, 24, 25))
        if rng.random() < 0.7:
            top = {0: 21, 24: 21, 25: 17}[query]
            return {"kind": "match", "graph": "rmat", "size": rng.randint(9, top), "factor": rng.choice((8, 12, 16)),
                    "query": query, "per_root": False}
        return {"kind": "match", "graph": "social", "size": log_size(rng, 3000, 200000), "query": query,
                "per_root": False}
    if kind == "pattern":
        # patterns that are no cliques, and cliques with a count per root
        query = rng.choice((1, 2, 5, 7, 8, 9, 12, 24))
        top = {1: 5000, 2: 100000, 9: 20000, 12: 4000, 24: 100000}.get(query, 6000)
        return {"kind": "match", "graph": "chunglu", "size": log_size(rng, 600, top), "query": query,
                "per_root": rng.random() < 0.5 or query == 24}
    if kind == "batch":
        largest = rng.choice((4, 5))
        return {"kind": "batch", "graph": "rmat", "size": rng.randint(6, 7 if largest == 5 else 9), "factor": 8,
                "queries": log_size(rng, 8, 96), "largest": largest}
    if kind == "mce":
        graph = rng.choice(("rmat", "chunglu", "social"))
        size = {"rmat": lambda: rng.randint(8, 11), "chunglu": lambda: log_size(rng, 1000, 150000),
                "social": lambda: log_size(rng, 3000, 300000)}[graph]()
        return {"kind": "mce", "graph": graph, "size": size, "per_root": rng.random() < 0.5}
    if kind == "view":
        return {"kind": "view", "graph": "rmat", "size": rng.randint(10, 18), "query": rng.choice((0, 24)),
                "bins": rng.choice((2, 3, 4))}
    if kind == "schedule":
        return {"kind": "schedule", "graph": "social", "size": log_size(rng, 3000, 200000)}
    return {"kind": "train", "rows": log_size(rng, 500, 50000), "epochs": rng.choice((1, 2, 3)),
            "batch": rng.choice((256, 512, 1024))}


# ---- graphs -------------------------------------------------------------------


def rmat(scale, factor, seed, isolated):
    """R-MAT graph drawn on the GPU: symmetrised; duplicates, self loops and (unless wanted) isolated vertices go"""
    n, m = 1 << scale, factor << scale
    rand = torch.Generator(device="cuda")
    rand.manual_seed(seed)
    u = torch.zeros(m, dtype=torch.int64, device="cuda")
    v = torch.zeros(m, dtype=torch.int64, device="cuda")
    for _ in range(scale):
        x = torch.rand(m, generator=rand, device="cuda", dtype=torch.float64)
        u = (u << 1) | (x >= 0.76)
        v = (v << 1) | (((x >= 0.57) & (x < 0.76)) | (x >= 0.95))
    perm = torch.randperm(n, generator=rand, device="cuda")
    u, v = perm[u], perm[v]
    keep = u != v
    u, v = u[keep], v[keep]
    key = torch.unique(torch.cat(((u << 32) | v, (v << 32) | u)))
    u, v = key >> 32, key & 0xFFFFFFFF
    deg = torch.bincount(u, minlength=n)
    held = torch.ones_like(deg, dtype=torch.bool) if isolated else deg > 0
    ids = torch.cumsum(held, 0) - 1
    row_ptrs = torch.zeros(int(held.sum()) + 1, dtype=torch.int64, device="cuda")
    row_ptrs[1:] = torch.cumsum(deg[held], 0)
    return g2.Graph(row_ptrs.cpu().numpy().view(np.uint64), ids[v].to(torch.int32).cpu().numpy().view(np.uint32))


def make_graph(case, seed):
    size = case["size"]
    # where every vertex has an output, isolated vertices stay: the outputs of a size then have one length
    isolated = case.get("per_root", False) or case["kind"] == "schedule"
    if case["graph"] == "rmat":
        return rmat(size, case.get("factor", 16), seed, isolated)
    if case["graph"] == "chunglu":
        w_max = min(2000.0, 6.32 * math.sqrt(size))  # 2000 at 100k vertices
        g = g2.gen_chung_lu(size, 2.3, 2.0, w_max, 10 * size, seed)
        return g if isolated else g.preprocess()
    f = size / 65e6
    w_max = min(5000.0, 3.4 * math.sqrt(size))  # hubs stay below the degree at which every pair of them is joined
    g = g2.gen_social(size, 2.1, 2.0, w_max, int(1.54e9 * f), int(2e6 * f), 10, 200, 3.0, 0.3, 0.9, 1e4, seed)
    return g if isolated else g.preprocess()


# ---- one case -----------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        rng = np.random.default_rng(seed)
        x = rng.standard_normal((case["rows"], 8)).astype(np.float32)
        y = (3.0 + x @ np.linspace(1.0, -0.5, 8) + 0.5 * np.maximum(x[:, 0] * x[:, 3], 0.0)
             + 0.1 * rng.standard_normal(case["rows"]))
        return {"kind": kind, "case": case, "x": x, "y": y.astype(np.float32),
                "mlp": device.Mlp(device=0, seed=1 + seed % 1000)}
    g = make_graph(case, seed)
    ex = g2.Executor(device=0)
    state = {"kind": kind, "case": case, "ex": ex}
    if kind == "match":
        ex.transfer(g)
        ex.set_plan(g2.plan_for_preset(case["query"]))
    elif kind == "batch":
        ex.transfer(g)
        queries = batch.random_queries(g2, case["queries"], seed, nmax=case["largest"])
        order = batch.heavy_first(queries)
        state.update(plans=[g2.plan_build(q) for q in queries], order=order)
    elif kind == "mce":
        ex.transfer(g.kcore_recode()[0])
    elif kind == "view":
        plan = g2.plan_for_preset(case["query"])
        sources = np.arange(seed % case["bins"], g.nv, case["bins"], dtype=np.uint32)
        state.update(graph=g2.view_materialize(g, sources, plan.hop, plan.root_degree), sources=sources)
        ex.set_plan(plan)
    else:
        g, _, shells, _ = g.kcore_recode()
        ex.transfer(g)
        core = np.repeat(np.arange(len(shells) - 1, dtype=np.uint32), np.diff(shells).astype(np.int64))
        rng = np.random.default_rng(seed)
        # a cost model's parameters: W1, b1, W2, b2, W3, b3, and the inputs' means and scales
        params = np.concatenate((rng.normal(0, 0.5, 512), np.zeros(64), rng.normal(0, 0.18, 4096), np.zeros(64),
                                 rng.normal(0, 0.25, 64), [3.0])).astype(np.float32)
        mlp = device.Mlp(device=0, seed=1)
        mlp.set_params(params)
        state.update(mlp=mlp, core=core, mu=np.array([3.5, 3.0, 7.0, 4.5, 0.3, 0.5, 0.8, 2.5], np.float32),
                     sd=np.array([1.0, 0.8, 1.5, 2.0, 0.2, 0.3, 0.3, 1.0], np.float32))
    return state


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "match":
        r = state["ex"].run_gm(per_root=case["per_root"])
        return [r["count"], r["per_root_count"]] if case["per_root"] else [r["count"]]
    if kind == "batch":
        r = state["ex"].run_gm_batch(state["plans"], order=state["order"])
        return [r["counts"]]
    if kind == "mce":
        r = state["ex"].run_mce(per_root=case["per_root"])
        return [r["total"], r["hist"]] + ([r["per_root_nodes"]] if case["per_root"] else [])
    if kind == "view":
        state["ex"].transfer(state["graph"], state["sources"])
        return [state["ex"].run_gm()["count"]]
    if kind == "schedule":
        return list(state["ex"].learned_schedule(state["mlp"], state["mu"], state["sd"], WAVES, core=state["core"]))
    loss = state["mlp"].train(state["x"], state["y"], epochs=case["epochs"], batch=case["batch"], lr=2e-3)
    return [loss, state["mlp"].params()]


def work(case):
    """Every case reads its graph once (row offsets 8 B, columns 4 B each way, sources 4 B) and writes its
    outputs; a schedule also reads 64 registers per vertex once and runs the cost model, a training call
    reads its rows once per epoch and does three products per layer."""
    weights = 8 * 64 + 64 * 64 + 64
    if case["kind"] == "train":
        rows = case["rows"] * case["epochs"]
        return {"bytes": 36 * rows + 4 * 4801, "flops": 6 * weights * rows}
    size = case["size"]
    if case["graph"] == "rmat":
        nv, ne = 1 << size, 2 * case.get("factor", 16) << size
    else:
        nv, ne = size, 20 * size if case["graph"] == "chunglu" else 55 * size
    need = 12 * nv + 4 * ne
    if case.get("per_root"):
        need += 8 * nv
    if case["kind"] == "schedule":
        return {"bytes": need + (64 + 12) * nv, "flops": 2 * weights * nv}
    if case["kind"] == "batch":
        return {"bytes": need + 8 * case["queries"], "flops": 0}
    return {"bytes": need + 8, "flops": 0}


def exact(case, seed):
    """Clique counts of small graphs, from dense adjacency matrices in 64 bits; None elsewhere."""
    if case["kind"] != "match" or case["query"] not in (0, 24) or case["per_root"]:
        return None
    if case["graph"] != "rmat" or case["size"] > 11:
        return None
    g = make_graph(case, seed)
    rows = np.repeat(np.arange(g.nv), g.degrees().astype(np.int64))
    a = torch.zeros((g.nv, g.nv), dtype=torch.float64, device="cuda")
    a[torch.from_numpy(rows).cuda(), torch.from_numpy(g.cols.astype(np.int64)).cuda()] = 1.0
    if case["query"] == 0:
        return [int((a * (a @ a)).sum().item()) // 6]
    total = 0.0
    for v in range(g.nv):  # triangles among the later neighbours of v
        later = g.cols[int(g.row_ptrs[v]):int(g.row_ptrs[v + 1])].astype(np.int64)
        later = torch.from_numpy(later[later > v]).cuda()
        b = a[later][:, later].contiguous()
        total += (b * (b @ b)).sum().item()
    return [int(total) // 6]
