"""The engine's kernels on the CPU: every program on small graphs under update
batches, its lists and results against the oracle, every access checked against
the allocation it falls in.

Odd batches hold what generated streams seldom do: deletes of edges that are not
there, also from sources without edges; deletes of the batch's own inserts.
"""
import numpy as np
import pytest

import oracle as O
import sgraph

PR_REL_TOL = 5e-5
HOST = sgraph.FLAG_HOST_EDGES


def graph(r, nv, per_vertex):
    """Two thirds of the sources may have edges, a few of them many."""
    ne = int(nv * per_vertex)
    s = np.where(r.random(ne) < 0.3, r.integers(0, max(1, nv // 50 + 1), ne), r.integers(0, nv, ne))
    s, d = np.where(s % 3 == 1, s // 2, s), r.integers(0, nv, ne)
    p = np.unique(np.stack([s, d], 1)[s != d], axis=0)
    row = np.zeros(nv + 1, np.uint64)
    np.cumsum(np.bincount(p[:, 0], minlength=nv), out=row[1:])
    return row, p[:, 1].astype(np.uint32)


def batch(r, nv, row, col, nins, ndel, odd):
    src = np.repeat(np.arange(nv), np.diff(row.astype(np.int64)))
    ins = r.integers(0, nv, (nins, 2))
    ins[:, 0] = np.where(r.random(nins) < 0.3, r.integers(0, nv), ins[:, 0])  # one source gains a third
    ins = ins[ins[:, 0] != ins[:, 1]]
    k = r.integers(0, len(col), ndel)
    dele = np.stack([src[k], col[k]], 1)
    if odd:
        dele = np.where((r.random(ndel) < 0.5)[:, None], r.integers(0, nv, (ndel, 2)), dele)
        dele = np.where((r.random(ndel) < 0.2)[:, None], ins[r.integers(0, len(ins), ndel)], dele)
    return ins.astype(np.uint32), dele.astype(np.uint32)


def check_lists(eng, row, col, tag):
    r, c = eng.adjacency()[:2]
    assert np.array_equal(np.asarray(r, np.uint64), row), f"{tag}: degrees"
    for v in range(len(row) - 1):
        a, b = int(row[v]), int(row[v + 1])
        assert np.array_equal(np.sort(c[a:b]), np.sort(col[a:b])), f"{tag}: list of {v}"


def check_values(eng, algo, queries, row, col, tag):
    if algo == "multi":
        for q in range(0, len(queries), max(1, len(queries) // 6)):
            kind, s = queries[q]
            exp = O.bfs(row, col, s) if kind == "bfs" else O.sssp(row, col, s, "seeded", 7)
            assert np.array_equal(eng.query(q), exp), f"{tag}: query {q}"
        return
    if algo in ("pr", "prcc"):
        exp = O.pagerank(row, col)
        rel = np.max(np.abs((eng.query(0) if algo == "prcc" else eng.values()).astype(np.float64) - exp) / exp)
        assert rel <= PR_REL_TOL, f"{tag}: rel {rel}"
    if algo == "prcc":
        assert np.array_equal(eng.query(1), O.cc(row, col)), tag
    elif algo != "pr":
        exp = O.cc(row, col) if algo == "cc" else O.bfs(row, col, 0) if algo == "bfs" else O.sssp(row, col, 0, "seeded", 7)
        assert np.array_equal(eng.values(), exp), tag


def run(algo, nv, per_vertex, sizes, seed, nq=0, odd=False, **cfg):
    r = np.random.default_rng(seed)
    row, col = graph(r, nv, per_vertex)
    queries = [(["bfs", "sssp"][i % 2], int(r.integers(0, nv))) for i in range(nq)]
    eng = sgraph.Engine(algo, weight_mode="seeded", weight_seed=7, round_blocks=8, **cfg)
    try:
        eng.load_csr(row, col)
        if algo == "multi":
            eng.init_queries(np.array([s for _, s in queries], np.uint32), [k for k, _ in queries])
        else:
            eng.init(0 if algo in ("bfs", "sssp") else None)
        check_values(eng, algo, queries, row, col, "G0")
        for t, (nins, ndel) in enumerate(sizes):
            ins, dele = batch(r, nv, row, col, nins, ndel, odd)
            eng.apply(ins, dele)
            row, col = O.apply_updates(row, col, ins, dele)
            check_lists(eng, row, col, f"G{t + 1}")
            check_values(eng, algo, queries, row, col, f"G{t + 1}")
    finally:
        eng.close()


SIZES = [(400, 400), (5, 40), (2500, 2500)]


@pytest.mark.parametrize("density,odd", [(0.25, False), (0.25, True), (1.0, False), (1.0, True)])
@pytest.mark.parametrize("algo,cfg", [
    ("bfs", {}), ("sssp", dict(flags=sgraph.FLAG_IN_EDGES)), ("cc", {}), ("cc", dict(flags=HOST, segments=5, cache_level=4)),
    ("pr", {}), ("pr", dict(pull_divisor=sgraph.PULL_ALWAYS)), ("pr", dict(pull_divisor=sgraph.PULL_NEVER)),
    ("prcc", dict(flags=HOST, segments=5, edge_budget_gb=2e-5)),
])
def test_programs(emulated, algo, cfg, density, odd):
    run(algo, 700, 5, SIZES, seed=31, odd=odd, pma_density=density, **cfg)


def test_streamed_pulls(emulated):
    run("pr", 200, 5, SIZES[:2], seed=33, flags=HOST | sgraph.FLAG_PULL_STREAM, segments=2, pull_divisor=sgraph.PULL_ALWAYS)


@pytest.mark.parametrize("density,odd", [(0.25, False), (0.25, True), (1.0, True)])
@pytest.mark.parametrize("nq", [3, 20, 70])  # one light group, one group of 32, two of 64
def test_batched_queries(emulated, nq, density, odd):
    run("multi", 700, 5, SIZES, seed=32, nq=nq, odd=odd, pma_density=density)
