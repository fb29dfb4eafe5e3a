"""The workloads this engine is timed on.

A streaming-graph program loads a graph, solves its vertex program once, then
applies one snapshot of edge inserts and deletes after another and reads the
results. The cases are those calls through the Python binding of the C ABI:

  stream   one engine (PageRank, SSSP, BFS, CC, or PageRank + CC on shared
           stores): a pass applies a snapshot and reads its results, then
           applies the snapshot that takes it back and reads again. The graph
           is the same before and after, so passes repeat.
  solve    the static solve from nothing (sg_init) and its results.
  queries  batched BFS / SSSP queries on one graph: a pass is as in "stream",
           reading some of the queries, or ("solve": True) starts the whole
           batch afresh.
  lookup   pointwise reads of a standing result, as a serving loop does them.

Graphs are R-MAT with the generator's usual quadrant probabilities, drawn here
with torch from the seed alone; self-loops and duplicates are dropped. "nv"
need not be a power of two (ids past it are dropped), "permute" gives the
vertices random ids, "hub" draws that share of the inserts from the 1 % of
sources with the most out-edges.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "c-gpustreamgraph_amd"))

import sgraph  # noqa: E402

A, B, C = 0.57, 0.19, 0.19
DAMPING = 0.85


def listed():
    return [
        # a serving loop's smallest call: a few thousand standing levels of a BFS
        dict(name="lookup_4k_of_256k", kind="lookup", algo="bfs", nv=262144, ef=16, n=4096),
        # small graph, small batches: the latency of launches and waits
        dict(name="bfs_64k_1k", kind="stream", algo="bfs", nv=65536, ef=16, ins=1000, dele=1000),
        # PageRank at the smallest configuration: scale 16, 10k + 10k per snapshot
        dict(name="pr_64k_10k", kind="stream", algo="pr", nv=65536, ef=16, ins=10000, dele=10000),
        # component labels kept on a graph of ragged size with random ids, with the in-edge store
        dict(name="cc_1m_ragged_in", kind="stream", algo="cc", nv=1000003, ef=12, ins=30011, dele=20011, permute=True,
             in_edges=True),
        # the incremental SSSP configuration: scale 22, 100k + 100k, seeded weights
        dict(name="sssp_4m_100k", kind="stream", algo="sssp", nv=4194304, ef=16, ins=100000, dele=100000,
             weights="seeded"),
        # PageRank kept on a middling graph of ragged size with random ids
        dict(name="pr_1m5_50k", kind="stream", algo="pr", nv=1500007, ef=24, ins=50021, dele=50021, permute=True),
        # PageRank on a large resident graph (200 M edges), a big batch
        dict(name="pr_8m_500k", kind="stream", algo="pr", nv=8388608, ef=24, ins=500000, dele=500000),
        # the static PageRank solve that every PageRank program starts with
        dict(name="pr_solve_4m", kind="solve", algo="pr", nv=4194304, ef=16),
        # the static SSSP solve over all edges, weights from the hash
        dict(name="sssp_solve_4m", kind="solve", algo="sssp", nv=4194304, ef=16, weights="hash128"),
        # 64 BFS + 64 SSSP standing queries kept under a batch
        dict(name="queries_128_1m_30k", kind="queries", nv=1048576, ef=16, ins=15000, dele=15000, queries=128, read=2,
             solve=False),
        # a batch of queries answered from nothing
        dict(name="queries_solve_64_512k", kind="queries", nv=524288, ef=16, ins=0, dele=0, queries=64, read=8,
             solve=True),
        # PageRank + CC out of memory: edge arrays in pinned host memory, most in-edges copied in HBM, hub-biased inserts
        dict(name="prcc_host_2m_50k", kind="stream", algo="prcc", nv=2097152, ef=16, ins=50000, dele=50000, hub=0.8,
             host_gb=0.07, density=0.6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stream"] * 5 + ["solve"] * 2 + ["queries"] * 2 + ["lookup"])
    nv = _log(rng, 50000, 6000000)
    ef = rng.randint(8, 24)
    if kind == "lookup":
        return dict(kind=kind, algo=rng.choice(["bfs", "cc", "pr"]), nv=min(nv, 2000003), ef=ef, n=_log(rng, 64, 60000))
    if kind == "solve":
        algo = rng.choice(["pr", "sssp", "bfs", "cc"])
        return dict(kind=kind, algo=algo, nv=nv, ef=ef, weights=rng.choice(["seeded", "hash128"]),
                    permute=rng.random() < 0.5)
    if kind == "queries":
        nv = min(nv, 1000003)
        b = _log(rng, 500, 60000)
        return dict(kind=kind, nv=nv, ef=ef, ins=b, dele=b + 7, queries=rng.choice([8, 33, 64, 100, 128]), read=2,
                    solve=rng.random() < 0.3)
    algo = rng.choice(["pr", "pr", "sssp", "bfs", "cc", "prcc"])
    b = _log(rng, 300, min(300000, nv // 8))
    c = dict(kind=kind, algo=algo, nv=nv, ef=ef, ins=b, dele=max(1, b - rng.randint(0, b // 2)),
             permute=rng.random() < 0.5, hub=rng.choice([0.0, 0.0, 0.8]))
    if algo == "sssp":
        c["weights"] = rng.choice(["seeded", "hash128", "one"])
    if algo in ("sssp", "bfs", "cc"):
        c["in_edges"] = rng.random() < 0.4
    return c


# ---- inputs -----------------------------------------------------------------
def _rmat(n, bits, gen):
    """n R-MAT draws as (source, target), int64."""
    src = torch.zeros(n, dtype=torch.int64, device="cuda")
    dst = torch.zeros(n, dtype=torch.int64, device="cuda")
    for _ in range(bits):
        x = torch.rand(n, generator=gen, device="cuda")
        src.mul_(2).add_(x >= A + B)
        dst.mul_(2).add_(((x >= A) & (x < A + B)) | (x >= A + B + C))
    return src, dst


def _inputs(case, seed):
    """Sorted edge keys (source << 32 | target) of the graph, the inserts (new
    edges) and deletes (edges of the graph) as key tensors, and the generator."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 1000003 + 17)
    nv = case["nv"]
    bits = max(1, (nv - 1).bit_length())
    perm = torch.randperm(nv, generator=gen, device="cuda") if case.get("permute") else None

    def pairs(n):
        s, d = _rmat(n, bits, gen)
        ok = (s < nv) & (d < nv) & (s != d)
        s, d = s[ok], d[ok]
        if perm is not None:
            s, d = perm[s], perm[d]
        return s, d

    # ragged sizes: draw as many edges as the power of two would have
    s, d = pairs(nv * case["ef"])
    keys = torch.unique((s << 32) | d)
    del s, d
    ins = dele = None
    n_ins, n_del = case.get("ins", 0), case.get("dele", 0)
    if n_ins:
        s, d = pairs(4 * n_ins + 1024)
        hub = case.get("hub", 0.0)
        if hub:
            deg = torch.bincount(keys >> 32, minlength=nv)
            top = torch.topk(deg, max(1, nv // 100)).indices
            pick = top[torch.randint(top.numel(), s.shape, generator=gen, device="cuda")]
            s = torch.where(torch.rand(s.shape, generator=gen, device="cuda") < hub, pick, s)
        k = torch.unique(((s << 32) | d)[s != d])
        at = torch.searchsorted(keys, k).clamp_(max=keys.numel() - 1)
        k = k[keys[at] != k]
        ins = k[torch.randperm(k.numel(), generator=gen, device="cuda")[:n_ins]]
    if n_del:
        at = torch.unique(torch.randint(keys.numel(), (n_del + n_del // 4 + 64,), generator=gen, device="cuda"))
        at = at[torch.randperm(at.numel(), generator=gen, device="cuda")[:n_del]]
        dele = keys[at]
    return keys, ins, dele, gen


def _csr(nv, keys):
    row = torch.searchsorted(keys, torch.arange(nv + 1, device="cuda", dtype=torch.int64) << 32)
    return row.cpu().numpy().astype(np.uint64), (keys & 0xFFFFFFFF).to(torch.int32).cpu().numpy().view(np.uint32)


def _pairs(keys):
    if keys is None:
        return np.zeros((0, 2), dtype=np.uint32)
    return torch.stack([keys >> 32, keys & 0xFFFFFFFF], 1).to(torch.int32).cpu().numpy().view(np.uint32)


def _ints(gen, hi, n):
    return torch.randint(hi, (n,), generator=gen, device="cuda").cpu().numpy().astype(np.uint32)


def _source(row, gen):
    """A source that reaches much of the graph: of 64 random vertices the one with the most out-edges."""
    some = _ints(gen, len(row) - 1, 64).astype(np.int64)
    return int(some[np.argmax(row[some + 1] - row[some])])


def prepare(case, seed):
    keys, ins, dele, gen = _inputs(case, seed)
    row, col = _csr(case["nv"], keys)
    del keys
    cfg = {}
    if case.get("weights"):
        cfg.update(weight_mode=case["weights"], weight_seed=int(seed) + 5)
    if case.get("in_edges"):
        cfg["flags"] = sgraph.FLAG_IN_EDGES
    if case.get("host_gb"):
        cfg.update(flags=sgraph.FLAG_HOST_EDGES, edge_budget_gb=case["host_gb"], cache_level=0, segments=16)
    if case.get("density"):
        cfg["pma_density"] = case["density"]
    st = {"case": case, "ins": _pairs(ins), "dele": _pairs(dele)}
    if case["kind"] == "queries":
        nq = case["queries"]
        eng = sgraph.Engine("multi", weight_mode="seeded", weight_seed=int(seed) + 5)
        eng.load_csr(row, col)
        st["sources"] = _ints(gen, case["nv"], nq)
        st["kinds"] = ["bfs"] * (nq // 2) + ["sssp"] * (nq - nq // 2)
        st["read"] = [i * (nq - 1) // max(1, case["read"] - 1) for i in range(case["read"])]
        if not case["solve"]:
            eng.init_queries(st["sources"], st["kinds"])
    else:
        eng = sgraph.Engine(case["algo"], **cfg)
        eng.load_csr(row, col)
        st["source"] = _source(row, gen) if case["algo"] in ("bfs", "sssp") else None
        if case["kind"] != "solve":
            eng.init(st["source"])
        if case["kind"] == "lookup":
            st["ids"] = _ints(gen, case["nv"], case["n"])
    st["eng"] = eng
    return st


# ---- one pass -----------------------------------------------------------------
def _results(eng, algo):
    return [eng.query(0), eng.query(1)] if algo == "prcc" else [eng.values()]


def run(st):
    case, eng = st["case"], st["eng"]
    kind = case["kind"]
    if kind == "lookup":
        got = eng.gather_at(st["ids"])
        return got.view(np.float32) if case["algo"] == "pr" else got
    if kind == "solve":
        eng.init(st["source"])
        return _results(eng, case["algo"])
    if kind == "queries" and case["solve"]:
        eng.init_queries(st["sources"], st["kinds"])
        return [eng.query(q) for q in st["read"]]
    out = []
    for ins, dele in ((st["ins"], st["dele"]), (st["dele"], st["ins"])):
        eng.apply(ins, dele)
        out.append([eng.query(q) for q in st["read"]] if kind == "queries" else _results(eng, case["algo"]))
    return out


def work(case):
    """Bytes: the live edges' ids once per snapshot or solve (4 B each: the edges
    into reset vertices can be any of them, PageRank's residuals travel along
    all), 12 B of state per vertex (and query), the batch (8 B a pair, and the
    list entry it changes), and the results read back."""
    nv, ne = case["nv"], case["nv"] * case["ef"]
    if case["kind"] == "lookup":
        return {"bytes": 12 * case["n"], "flops": 0}
    nq = case.get("queries", 1)
    reads = case["read"] if case["kind"] == "queries" else 2 if case["algo"] == "prcc" else 1
    one = 4 * ne + 12 * nv * nq + 4 * nv * reads
    fl = 2 * ne if case.get("algo") in ("pr", "prcc") else 0
    if case["kind"] == "solve" or case.get("solve"):
        return {"bytes": one, "flops": fl}
    return {"bytes": 2 * (one + 16 * (case["ins"] + case["dele"])), "flops": 2 * fl}


# ---- 64-bit results --------------------------------------------------------------
def _pagerank(nv, keys):
    """Fixed point of r = (1 - a) + a * sum over in-edges of r(u) / outdeg(u), in float64."""
    u, v = keys >> 32, keys & 0xFFFFFFFF
    deg = torch.bincount(u, minlength=nv).clamp_(min=1).double()
    order = torch.argsort(v, stable=True)
    u, v = u[order], v[order]
    end = torch.searchsorted(v, torch.arange(nv + 1, device="cuda"))
    total = torch.zeros(u.numel() + 1, dtype=torch.float64, device="cuda")
    r = torch.full((nv,), 1.0 - DAMPING, dtype=torch.float64, device="cuda")
    for _ in range(400):
        torch.cumsum((r / deg)[u], 0, out=total[1:])
        new = (1.0 - DAMPING) + DAMPING * (total[end[1:]] - total[end[:-1]])
        move = float((new - r).abs().max())
        r = new
        if move < 1e-12:
            break
    return r.cpu().numpy()


def exact(case, seed):
    """PageRank's ranks in float64 (levels, distances and labels are whole numbers)."""
    if case.get("algo") not in ("pr", "prcc"):
        return None
    keys, ins, dele, gen = _inputs(case, seed)
    if case["kind"] == "lookup":
        return _pagerank(case["nv"], keys)[_ints(gen, case["nv"], case["n"]).astype(np.int64)]
    if case["kind"] == "solve":
        return [_pagerank(case["nv"], keys)]
    kept = keys[~torch.isin(keys, dele, assume_unique=True)]
    after = torch.sort(torch.cat([kept, ins])).values
    both = [_pagerank(case["nv"], after), _pagerank(case["nv"], keys)]
    return [[r, None] if case["algo"] == "prcc" else [r] for r in both]
