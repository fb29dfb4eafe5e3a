"""Update batches at the sizes and mixes where their sort can go wrong: one
bucket, the first size past it, many buckets, the largest size sorted in
buckets and the first past it; one source for every insert, one pair for every
delete, runs of a few pairs, ids past nv. Adjacency sequences (file order per
source) equal the oracle's update model.
"""
import numpy as np
import pytest

import oracle as O
import sgraph

pytestmark = pytest.mark.gpu

NV = 5000


def graph(seed):
    rng = np.random.default_rng(seed)
    u = rng.integers(0, NV, 30000)
    u[:8000] = 7  # a hub
    pairs = np.unique(np.stack([u, rng.integers(0, NV, 30000)], 1), axis=0)
    row = np.zeros(NV + 1, dtype=np.uint64)
    np.cumsum(np.bincount(pairs[:, 0], minlength=NV).astype(np.uint64), out=row[1:])
    return row, pairs[:, 1].astype(np.uint32), pairs.astype(np.uint32)


def batch(mix, n, pairs, seed):
    rng = np.random.default_rng(seed)
    ins = rng.integers(0, NV, (n, 2)).astype(np.uint32)
    dele = pairs[rng.integers(0, len(pairs), n)]
    if mix == "one":  # one source of all inserts, one pair of all deletes
        ins[:, 0] = 11
        dele = np.repeat(pairs[5:6], n, axis=0)
    elif mix == "runs":  # a few pairs over and over, in an order that repeats
        ins = ins[np.arange(n) % 37]
        dele = pairs[(np.arange(n) % 53) * 101]
    return ins, np.ascontiguousarray(dele)


@pytest.mark.parametrize("mix", ["random", "one", "runs"])
@pytest.mark.parametrize("n", [1, 2, 1023, 2048, 2049, 3000, 40000, 1 << 20, (1 << 20) + 1])
def test_batch(mix, n):
    if n > 50000 and mix == "one":
        n = min(n, 1 << 20)
    row, col, pairs = graph(3)
    ins, dele = batch(mix, n, pairs, n)
    e = sgraph.Engine("bfs")
    try:
        e.load_csr(row, col)
        e.init(0)
        e.apply(ins, dele)
        r, c = O.apply_updates(row, col, ins, dele)
        gr, gc = e.adjacency()[:2]
        assert np.array_equal(gr, r), "degrees differ"
        assert np.array_equal(gc, c), "adjacency sequences differ"
        assert np.array_equal(e.values(), O.bfs(r, c, 0))
    finally:
        e.close()


@pytest.mark.parametrize("n", [500, 9000])
def test_dropped_pairs(n):
    row, col, pairs = graph(4)
    ins, dele = batch("random", n, pairs, 5)
    bad_i, bad_d = ins.copy(), dele.copy()
    bad_i[::7, 0] = NV + 3
    bad_i[3::7, 1] = 0xFFFFFFFF
    bad_d[::5, 1] = NV
    keep_i, keep_d = np.all(bad_i < NV, 1), np.all(bad_d < NV, 1)
    e = sgraph.Engine("bfs")
    try:
        e.load_csr(row, col)
        e.init(0)
        e.apply_device(e.to_device(bad_i), n, e.to_device(bad_d), n)
        r, c = O.apply_updates(row, col, bad_i[keep_i], bad_d[keep_d])
        gr, gc = e.adjacency()[:2]
        assert np.array_equal(gr, r) and np.array_equal(gc, c)
        assert e.stats()["dropped_updates"] == int((~keep_i).sum() + (~keep_d).sum())
    finally:
        e.close()
