"""Batches whose deletes remove nothing ahead of the batch's inserts.

A source takes inserts and deletes in one batch. Where no delete hits its old
list (the edge is not there, or is one of the batch's own inserts), an insert
that survives keeps its place in the sequence old list ++ inserts, past the
list's end: it still has to be stored there. Lists are compared entry by entry
with the oracle, and batched queries walk them.
"""
import numpy as np
import pytest

import oracle as O
import sgraph

OLD = (0, 1, 5, 63, 64, 65, 130)  # entries before the batch
NEW = (1, 2, 63, 64, 65, 129)     # inserts
# what the deletes of a source are: an absent edge, the batch's first or last
# insert, the first or last entry of the old list
MISS = ("absent", "first new", "last new", "first old", "last old")


def workload():
    """A graph with one source for each combination, the batch, and what follows it."""
    cases = [(d, k, m) for d in OLD for k in NEW for m in MISS if d or "old" not in m]
    nv = 4 * len(cases)
    deg = np.zeros(nv, np.int64)
    src = np.arange(len(cases)) * 4 + 1  # sources apart from each other
    cols, ins, dele = [], [], []
    for s, (d, k, m) in zip(src, cases):
        t = (s * 7 + 3 * np.arange(d + k + 1)) % nv  # distinct targets: old, new, and one that stays absent
        deg[s] = d
        cols.append(t[:d])
        ins += [(s, x) for x in t[d:d + k]]
        at = {"absent": d + k, "first new": d, "last new": d + k - 1, "first old": 0, "last old": d - 1}[m]
        dele.append((s, t[at]))
    row = np.zeros(nv + 1, np.uint64)
    np.cumsum(deg, out=row[1:])
    back = [(x, y) for (x, y) in dele]  # the deleted ones come again while others go
    return (nv, row, np.concatenate(cols).astype(np.uint32), src,
            [(np.array(ins, np.uint32), np.array(dele, np.uint32)),
             (np.array(back, np.uint32), np.array(ins[::3], np.uint32))])


def apply_and_check(eng, row, col, batches):
    for t, (ins, dele) in enumerate(batches):
        eng.apply(ins, dele)
        row, col = O.apply_updates(row, col, ins, dele)
        r, c = eng.adjacency()[:2]
        assert np.array_equal(np.asarray(r, np.uint64), row), f"G{t + 1}: degrees"
        assert np.array_equal(c, col), f"G{t + 1}: lists, first at entry {int(np.argmax(c != col))}"
    return row, col


@pytest.mark.parametrize("density", [0.05, 0.25])  # most lists have room for the batch, some do not
@pytest.mark.parametrize("algo", ["bfs", "cc", "pr"])
def test_lists(backend, algo, density):
    nv, row, col, src, batches = workload()
    eng = sgraph.Engine(algo, pma_density=density, round_blocks=8)
    try:
        eng.load_csr(row, col)
        eng.init(int(src[0]) if algo == "bfs" else None)
        row, col = apply_and_check(eng, row, col, batches)
        got = eng.values()
        if algo == "pr":
            exp = O.pagerank(row, col)
            assert np.max(np.abs(got.astype(np.float64) - exp) / exp) <= 5e-5
        else:
            assert np.array_equal(got, O.cc(row, col) if algo == "cc" else O.bfs(row, col, int(src[0])))
    finally:
        eng.close()


@pytest.mark.parametrize("nq", [16, 17, 70])  # one light group, one group of 32, two of 64
def test_batched_queries(backend, nq):
    nv, row, col, src, batches = workload()
    sources = src[:: max(1, len(src) // nq)][:nq].astype(np.uint32)
    eng = sgraph.Engine("multi", weight_mode="seeded", weight_seed=7, pma_density=0.05, round_blocks=8)
    try:
        eng.load_csr(row, col)
        eng.init_queries(sources, ["bfs", "sssp"] * (len(sources) // 2) + ["bfs"] * (len(sources) % 2))
        row, col = apply_and_check(eng, row, col, batches)
        for q in range(len(sources)):
            exp = O.sssp(row, col, int(sources[q]), "seeded", 7) if q % 2 else O.bfs(row, col, int(sources[q]))
            assert np.array_equal(eng.query(q), exp), f"query {q}"
    finally:
        eng.close()
