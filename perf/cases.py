"""Performance cases: what a user of ripples_amd has it do, through its public entry points.

A case is a plain dict.  Its graph is a directed R-MAT graph (a/b/c/d = .57/.19/.19/.05,
duplicates and self loops removed) of any number of vertices, made on the GPU from the seed
alone: another seed is another graph, other weights and another sampling stream.

  op        imm      rip_imm on a resident graph: the whole call
            pool     an RRR pool filled and selected from: reset, sample, select
            export   an RRR pool filled and read back: reset, sample, export
            select   a resident pool queried: select, coverage of the seeds, occurrence counts
            opimc    rip_opimc on a resident graph: the whole call
            spread   Monte Carlo spread of a seed set
            serve    a batch of IMM queries on two resident graphs through the server
  weights   uniform  IC, w ~ U[0, wscale]            cascade  IC, w = 1 / indeg
            const    IC, w = wscale                  lt_norm  LT, in-weights normalised to wscale

Outputs are seed lists, RRR sets, counts and run records: whole numbers, apart from the
records' coverage fractions and bounds, which are quotients of them.  Lists whose length
depends on the seed (rounds of a run, seeds that cover anything, set members) come padded
with -1 to a length the case fixes.
"""
import math

import numpy as np
import torch

import ripples_amd as R

SERVE_K = (10, 50, 100, 200)
SERVE_EPS = (0.5, 0.2, 0.13)

# Mean RRR set sizes, for work() of resident pools (weighted cascade, LT normalised to 0.9).
MEAN_SET = {"cascade": 20, "lt_norm": 5}


def listed():
    return [
        # the smallest call: a user trying the tool on a small network, where launches,
        # synchronisations and allocations are all there is
        dict(name="imm_small", op="imm", n=1000, edge_factor=8, weights="cascade", wscale=1.0,
             k=5, eps=0.5),
        # IMM under IC with uniform weights, the sets that reach a giant component
        dict(name="imm_uniform_65k", op="imm", n=65536, edge_factor=16, weights="uniform",
             wscale=0.1, k=50, eps=0.5),
        # the same on the largest uniform graph of the serving mix
        dict(name="imm_uniform_262k", op="imm", n=262144, edge_factor=16, weights="uniform",
             wscale=0.1, k=10, eps=0.5),
        # IMM under LT at a million vertices
        dict(name="imm_lt_1m", op="imm", n=1048576, edge_factor=16, weights="lt_norm", wscale=0.9,
             k=100, eps=0.13),
        # IMM under weighted cascade at four million vertices, with a sampler setting kept from
        # an earlier autotuning
        dict(name="imm_cascade_4m", op="imm", n=4194304, edge_factor=16, weights="cascade",
             wscale=1.0, k=200, eps=0.1, queue_cap=64, block=256, wave_stage=1),
        # one sampling step and a selection on the largest graph: sets of hundreds of
        # thousands of vertices, held in the column store
        dict(name="pool_uniform_16m", op="pool", n=16777216, edge_factor=16, weights="uniform",
             wscale=0.02, k=100, sets=20000),
        # RRR sets drawn for a user's own analysis: sampled and read back, an odd size
        dict(name="export_lt_300k", op="export", n=300007, edge_factor=16, weights="lt_norm",
             wscale=0.9, sets=100000),
        # queries against a pool that is already there (another k, FindCoverage, counts)
        dict(name="select_cascade_1m", op="select", n=1048576, edge_factor=16, weights="cascade",
             wscale=1.0, k=100, sets=600000),
        # OPIM-C, the second driver of sampler and selector, with the default sampler setting
        dict(name="opimc_cascade_200k", op="opimc", n=200003, edge_factor=16, weights="cascade",
             wscale=1.0, k=50, eps=0.2),
        # the spread check of a seed set, as the simulator tool makes it, under both models
        dict(name="spread_uniform_262k", op="spread", n=262144, edge_factor=16, weights="uniform",
             wscale=0.1, k=50, replicas=256),
        dict(name="spread_lt_100k", op="spread", n=100003, edge_factor=16, weights="lt_norm",
             wscale=0.9, k=20, replicas=256),
        # served queries: different k and epsilon, half of them on the same stream
        dict(name="serve_12_queries", op="serve", n=262144, edge_factor=16, weights="cascade",
             wscale=1.0, queries=12),
    ]


def draw(rng):
    """One more case of the same ranges."""
    def size(lo, hi):
        v = int(2 ** rng.uniform(math.log2(lo), math.log2(hi)))
        return v if rng.random() < 0.3 else v | 1

    op = rng.choice(["imm", "imm", "imm", "pool", "export", "select", "opimc", "spread", "serve"])
    ef = rng.choice([4, 8, 16, 16, 24])
    weights = rng.choice(["uniform", "const", "cascade", "cascade", "lt_norm", "lt_norm"])
    if op in ("select", "export", "serve"):
        weights = "cascade" if op == "serve" else rng.choice(["cascade", "lt_norm"])
    giant = weights in ("uniform", "const")
    wscale = {"uniform": rng.uniform(0.02, 0.1), "const": rng.uniform(0.01, 0.04),
              "cascade": 1.0, "lt_norm": rng.uniform(0.5, 0.95)}[weights]
    c = dict(op=op, edge_factor=ef, weights=weights, wscale=round(wscale, 4))
    if op == "imm":
        c.update(n=size(500, 1 << 17 if giant else 1 << 21), k=rng.randint(1, 200),
                 eps=0.5 if giant else rng.choice(SERVE_EPS))
    elif op == "pool":
        c.update(n=size(1 << 12, 1 << 20), k=rng.randint(1, 200),
                 sets=size(1000, 20000 if giant else 1000000))
    elif op == "export":
        c.update(n=size(1 << 12, 1 << 20), sets=size(500, 200000))
    elif op == "select":
        c.update(n=size(1 << 12, 1 << 20), k=rng.randint(1, 200), sets=size(10000, 1000000))
    elif op == "opimc":
        c.update(n=size(1000, 1 << 16 if giant else 1 << 19), k=rng.randint(1, 100),
                 eps=0.4 if giant else rng.choice((0.4, 0.2)))
    elif op == "spread":
        c.update(n=size(1000, 1 << 18), k=rng.randint(1, 100), replicas=rng.randint(16, 256))
    else:
        c.update(n=size(1 << 14, 1 << 18), queries=rng.randint(2, 12))
    return c


def _edges(case):
    """Expected edges: draws less duplicates and self loops."""
    return int(0.94 * case["edge_factor"] * case["n"])


def work(case):
    """Bytes no implementation can do without: the inputs read once (the CSR, 8 per vertex and
    8 per edge, or the resident pool, 4 per member and 12 per set) and the outputs written
    once.  Drawing the sets itself has no such bound in terms of the case."""
    n, m = case["n"], _edges(case)
    csr = 8 * (n + 1) + 8 * m
    op = case["op"]
    if op == "select":
        pool = case["sets"] * (12 + 4 * MEAN_SET[case["weights"]])
        return {"bytes": pool + 4 * n + 4 * case["k"], "flops": 0}
    if op == "export":
        return {"bytes": csr + case["sets"] * (8 + 4 * MEAN_SET[case["weights"]]), "flops": 0}
    if op == "spread":
        return {"bytes": csr + 12 * case["replicas"], "flops": 0}
    if op == "serve":
        return {"bytes": 2 * csr + 4 * 100 * case["queries"], "flops": 0}
    return {"bytes": csr + 4 * case["k"], "flops": 0}


def _rmat(n, draws, gen):
    """Distinct (dst, src) keys dst * n + src of an R-MAT graph, ascending."""
    scale = max(1, (n - 1).bit_length())
    keys = []
    left = draws
    while left > 0:
        e = min(left, 1 << 26)
        left -= e
        src = torch.zeros(e, dtype=torch.int64, device="cuda")
        dst = torch.zeros(e, dtype=torch.int64, device="cuda")
        for _ in range(scale):
            u = torch.rand(e, generator=gen, device="cuda")
            s = u >= 0.76                                  # a + b
            d = ((u >= 0.57) & ~s) | (u >= 0.95)           # b, d
            src.mul_(2).add_(s)
            dst.mul_(2).add_(d)
        src, dst = (src * n) >> scale, (dst * n) >> scale  # any n, not only powers of two
        keys.append((dst * n + src)[src != dst])
        del src, dst, u, s, d
    key = torch.cat(keys)
    del keys
    return torch.unique(key)


def _host_csr(case, weights, seed):
    """Transposed CSR (in-neighbour rows) on the host, from the seed alone, and the vertices of
    largest out-degree, best first."""
    n = case["n"]
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    key = _rmat(n, case["edge_factor"] * n, gen)
    m = key.numel()
    dst = torch.div(key, n, rounding_mode="floor")
    src = key - dst * n
    del key
    deg = torch.bincount(dst, minlength=n)
    index = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    index[1:] = torch.cumsum(deg, 0)
    if weights == "cascade":
        w = 1.0 / deg[dst].to(torch.float32)
    elif weights == "const":
        w = torch.full((m,), case["wscale"], dtype=torch.float32, device="cuda")
    else:
        r = torch.randint(1, 1 << 24, (m,), generator=gen, device="cuda")
        if weights == "uniform":
            w = (r.to(torch.float64) * (case["wscale"] / (1 << 24))).to(torch.float32)
        else:
            run = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), torch.cumsum(r, 0)])
            row = run[index[1:]] - run[index[:-1]]         # integer row sums
            w = (r.to(torch.float64) * case["wscale"] / row[dst]).to(torch.float32)
            del run, row
        del r
    out = torch.bincount(src, minlength=n) * n + torch.arange(n - 1, -1, -1, device="cuda")
    best = torch.topk(out, min(n, 256)).indices.cpu().numpy().astype(np.uint32)
    host = (index.cpu().numpy().astype(np.uint64), src.to(torch.int32).cpu().numpy().view(np.uint32),
            w.cpu().numpy())
    del index, src, dst, deg, w, out
    torch.cuda.empty_cache()   # the library allocates beside torch
    return host, best


def _graph(case, weights, seed):
    (index, edges, w), best = _host_csr(case, weights, seed)
    return R.Graph(index, edges, w, model=R.LT if weights == "lt_norm" else R.IC), best


def _tune(case):
    t = {f: case[f] for f in ("queue_cap", "block", "wave_stage") if f in case}
    return t or None


def prepare(case, seed):
    """A resident graph and what else the program keeps: a pool, a seed set, queries."""
    g, best = _graph(case, case["weights"], seed)
    s = dict(case=case, graph=g, seed=int(seed), tune=_tune(case))
    op = case["op"]
    if op in ("pool", "export", "select"):
        s["pool"] = g.pool(int(seed))
    if op == "select":
        s["pool"].generate_rrr_sets(case["sets"])
    elif op == "export":
        # where the program collects the members
        s["vertices"] = np.full(5 * MEAN_SET[case["weights"]] * case["sets"], -1, np.int32)
    elif op == "spread":
        s["seeds"] = best[:case["k"]].copy()
    elif op == "serve":
        lt, _ = _graph(dict(case, wscale=0.9), "lt_norm", seed)
        s["graphs"] = [g, lt]
        s["queries"] = [(i % 2, SERVE_K[(i // 2) % 4], SERVE_EPS[(i // 3) % 3],
                         int(seed) if i % 4 < 2 else int(seed) + i) for i in range(case["queries"])]
    return s


def _padded(values, size, dtype):
    out = np.full(size, -1, dtype)
    out[:len(values)] = values
    return out


def _imm_out(case, seeds, rec):
    keep = ("Theta", "NumSets", "RRRElements", "Rounds", "LB", "FinalF")
    out = {k: rec[k] for k in keep}
    out["seeds"] = _padded(seeds, case["k"], np.int64)
    out["ThetaPrime"] = _padded(rec["ThetaPrime"], 64, np.int64)
    out["F"] = _padded(rec["F"], 64, np.float64)
    return out


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "imm":
        return _imm_out(c, *R.imm(s["graph"], c["k"], c["eps"], seed=s["seed"], tune=s["tune"]))
    if op == "opimc":
        seeds, rec = R.opimc(s["graph"], c["k"], c["eps"], seed=s["seed"])
        out = {k: rec[k] for k in ("ThetaZero", "ThetaMax", "Theta", "Rounds", "RRRElements")}
        for k in ("Coverage1", "Coverage2"):
            out[k] = _padded(rec[k], 64, np.int64)
        for k in ("Lower", "Upper", "Alpha"):
            out[k] = _padded(rec[k], 64, np.float32)
        out["seeds"] = _padded(seeds, c["k"], np.int64)
        return out
    if op == "spread":
        act, lev = s["graph"].spread(s["seeds"], c["replicas"], seed=s["seed"])
        return {"activated": act.astype(np.int64), "levels": lev}
    if op == "serve":
        srv = R.Server(slots=8, workers=4)
        try:
            ids = [srv.add_graph(g) for g in s["graphs"]]
            qs = [srv.submit(ids[gi], k, eps, seed) for gi, k, eps, seed in s["queries"]]
            done = [srv.poll(q) for q in qs]
        finally:
            srv.close()
        return {"seeds": [_padded(d[0], k, np.int64) for d, (_, k, _, _) in zip(done, s["queries"])],
                "Theta": np.array([d[1]["Theta"] for d in done], np.int64),
                "FinalF": np.array([d[1]["FinalF"] for d in done], np.float64)}
    pool = s["pool"]
    if op == "select":
        seeds, covered = pool.find_most_influential_set(c["k"])
        return {"seeds": _padded(seeds, c["k"], np.int64), "covered": covered,
                "coverage": pool.coverage(seeds),
                "counts": pool.count_occurrences()}
    pool.reset()
    pool.generate_rrr_sets(c["sets"], tune=s["tune"])
    if op == "export":
        off, ver = pool.export()
        s["vertices"][:len(ver)] = ver.view(np.int32)
        return {"offsets": off.astype(np.int64), "vertices": s["vertices"]}
    seeds, covered = pool.find_most_influential_set(c["k"])
    sets, elements = pool.size()
    return {"seeds": _padded(seeds, c["k"], np.int64), "covered": covered, "sets": sets,
            "elements": elements}


def exact(case, seed):
    """The outputs are samples of the library's own random streams and whole-number functions
    of them: no value in 64 bits stands for them."""
    return None
