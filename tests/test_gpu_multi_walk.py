"""Batched queries where the walk of a vertex's list can go wrong: lists that
end in, at or past a step of 64 edges and the chunk of 512, and every lane
layout of the active slots (4 or fewer, 8, 16, 32, all; one and two groups).

A hub reaches n vertices that form a chain back to it; queries start at the hub
and along the chain, so its list is walked for few and for many slots. Then
tree edges out of the hub go and come back. Distances equal the oracle's.
"""
import numpy as np
import pytest

import oracle as O
import sgraph

pytestmark = pytest.mark.gpu


def hub_graph(n):
    nv = n + 3
    src = [0] * n + list(range(1, n + 1))
    dst = list(range(1, n + 1)) + list(range(2, n + 2))
    src += [n + 1, n + 2, n + 1]
    dst += [n + 2, 0, 0]
    row = np.zeros(nv + 1, dtype=np.uint64)
    order = np.lexsort((dst, src))
    src, dst = np.array(src)[order], np.array(dst)[order]
    np.cumsum(np.bincount(src, minlength=nv).astype(np.uint64), out=row[1:])
    return nv, row, dst.astype(np.uint32)


@pytest.mark.parametrize("n", [3, 63, 64, 65, 511, 512, 513, 1100])
@pytest.mark.parametrize("nq", [3, 20, 40, 64, 70])
def test_hub_lists(n, nq):
    nv, row, col = hub_graph(n)
    rng = np.random.default_rng(1000 * n + nq)
    sources = np.where(rng.random(nq) < 0.5, 0, rng.integers(0, nv, nq)).astype(np.uint32)
    kinds = ["bfs" if i % 2 else "sssp" for i in range(nq)]
    gone = np.unique(rng.integers(1, n + 1, max(1, n // 5)))
    dele = np.stack([np.zeros(len(gone)), gone], 1).astype(np.uint32)
    none = np.zeros((0, 2), dtype=np.uint32)
    e = sgraph.Engine("multi", weight_mode="seeded", weight_seed=9)
    try:
        e.load_csr(row, col)
        e.init_queries(sources, kinds)
        r, c = row, col
        for step, (i, d) in enumerate([(none, none), (none, dele), (dele, none)]):
            if step:
                e.apply(i, d)
                r, c = O.apply_updates(r, c, i, d)
            for q in range(nq):
                exp = O.bfs(r, c, int(sources[q])) if kinds[q] == "bfs" else O.sssp(r, c, int(sources[q]), "seeded", 9)
                assert np.array_equal(e.query(q), exp), f"n={n} nq={nq} step {step} query {q}"
    finally:
        e.close()
