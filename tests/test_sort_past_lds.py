"""Batches whose sample sort leaves one bucket too large for LDS.

The sort takes its splitters from a sample, one pair of every few, at positions
that are known beforehand. Here the sampled pairs have one low source, so that
all the others, in any order, fall in the bucket past the last splitter, which
is then sorted in place. Lists equal the oracle's entry by entry.
"""
import numpy as np
import pytest

import oracle as O
import sgraph

NV = 3000
BUCKET, OVER, MOST_SPLIT, LDS = 768, 8, 512, 8192  # sg_sort.h: kSortBucket, kSortOver, kSortMaxSplit, kSortLds


def sampled(n):
    """Positions of the sample among n pairs (k_sort_count)."""
    ns = min(MOST_SPLIT, -(-n // BUCKET)) * OVER
    i = np.arange(ns, dtype=np.uint64)
    a, e = i * n // ns, (i + 1) * n // ns
    return (a + ((i * 2654435761 & 0xFFFFFFFF) >> 8) % (e - a)).astype(np.int64)


@pytest.mark.parametrize("side", ["inserts", "deletes", "both"])
@pytest.mark.parametrize("n", [9001, 16384, 20011])
def test_bucket_past_lds(backend, n, side):
    r = np.random.default_rng(n)
    at = sampled(n)
    k = r.permutation(1000 * NV)[:2 * n]  # distinct pairs of sources 1000 to 1999
    pairs = np.stack([1000 + k // NV, k % NV], 1)
    old, new = pairs[:n].copy(), pairs[n:].copy()
    for p, u in ((old, 3), (new, 4)):
        p[at] = np.stack([np.full(len(at), u), np.arange(len(at))], 1)
    assert n - len(at) > LDS
    order = np.lexsort((old[:, 1], old[:, 0]))
    row = np.zeros(NV + 1, np.uint64)
    np.cumsum(np.bincount(old[:, 0], minlength=NV), out=row[1:])
    col = old[order, 1].astype(np.uint32)
    ins, dele = new.astype(np.uint32), old.astype(np.uint32)
    if side == "inserts":
        dele = dele[:50]
    if side == "deletes":
        ins = ins[:50]
    eng = sgraph.Engine("bfs", round_blocks=8)
    try:
        eng.load_csr(row, col)
        eng.init(3)
        eng.apply(ins, dele)
        row, col = O.apply_updates(row, col, ins, dele)
        gr, gc = eng.adjacency()[:2]
        assert np.array_equal(np.asarray(gr, np.uint64), row) and np.array_equal(gc, col)
        assert np.array_equal(eng.values(), O.bfs(row, col, 3))
    finally:
        eng.close()
