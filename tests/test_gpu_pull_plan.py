"""PageRank pulls over the pull plan, at the sizes where its tiles can go wrong.

* In-lists of every size around a tile (512 in-edges): one list that ends in,
  at or past a tile boundary, one that spans many tiles, tiles full of
  one-edge lists, an edge count just below, at and above a multiple of 512, ids
  of 1 to 13 bits.
* A device budget with no room for the plan: it is given back, pulls read the
  store's slots, the results meet the same bounds.
* Rounds given up at max_rounds: the pushes under way are delivered, so a later
  update still reaches the fixed point of its graph.
Checked against the FP64 oracle within the bounds of the other PR tests
(5e-5 relative on raw ranks).
"""
import numpy as np
import pytest

import oracle as O
import sgraph

pytestmark = pytest.mark.gpu

PR_REL_TOL = 5e-5


def csr(nv, pairs):
    pairs = np.unique(np.asarray(pairs, dtype=np.int64).reshape(-1, 2), axis=0)
    row = np.zeros(nv + 1, dtype=np.uint64)
    np.cumsum(np.bincount(pairs[:, 0], minlength=nv).astype(np.uint64), out=row[1:])
    return row, pairs[:, 1].astype(np.uint32)


def check(eng, row, col, tag):
    exp = O.pagerank(row, col)
    rel = float(np.max(np.abs(eng.values().astype(np.float64) - exp) / exp))
    print(f"[gpu] plan {tag} rel={rel:.2e}", flush=True)
    assert rel <= PR_REL_TOL, f"{tag}: rel {rel}"


def star(n):  # one in-list of n edges
    return n + 1, [(u, 0) for u in range(1, n + 1)]


def ring(n):  # n in-lists of one edge
    return n, [(u, (u + 1) % n) for u in range(n)]


def mixed(n):  # lists of 1, 2, 3, ... edges up to n in all, and a long one after them
    nv, pairs, v, k = n + 600, [], 0, 1
    while len(pairs) < n:
        for j in range(min(k, n - len(pairs))):
            pairs.append(((v * 7 + j * 13 + 1) % nv, v))
        v, k = v + 2, k + 1
    pairs += [(u, nv - 1) for u in range(600)]
    return nv, [p for p in pairs if p[0] != p[1]]


@pytest.mark.parametrize("shape,n", [(star, n) for n in (1, 2, 511, 512, 513, 1024, 1500, 6000)] +
                         [(ring, n) for n in (2, 63, 512, 513, 1300)] + [(mixed, n) for n in (100, 512, 1023, 4000)])
def test_tiles_of_every_shape(shape, n):
    nv, pairs = shape(n)
    row, col = csr(nv, pairs)
    eng = sgraph.Engine("pr", pull_divisor=sgraph.PULL_ALWAYS)
    try:
        eng.load_csr(row, col)
        eng.init()
        check(eng, row, col, f"{shape.__name__} {n}")
        # two edges leave, one comes: list and tile boundaries shift
        src = np.repeat(np.arange(nv, dtype=np.uint32), np.diff(row.astype(np.int64)))
        dele = np.stack([src, col], 1)[[0, len(col) // 2]] if len(col) > 2 else np.zeros((0, 2), np.uint32)
        ins = np.array([[nv - 1, nv // 2]], dtype=np.uint32) if nv // 2 != nv - 1 else np.zeros((0, 2), np.uint32)
        eng.apply(ins, dele)
        r, c = O.apply_updates(row, col, ins, dele)
        check(eng, r, c, f"{shape.__name__} {n} updated")
        assert eng.stats()["pull_rounds"] > 0
    finally:
        eng.close()


def test_plan_given_back_under_a_device_budget():
    nv, row, col = sgraph.gen_rmat(13, 32, seed=95)
    ins, dele = sgraph.gen_updates(row, col, 13, 2, 2000, 2000, seed=96)
    whole, held = {}, None
    for budget in (0.0, None):
        if budget is None:  # less than the ids of the plan short
            budget = (held - len(col)) / 2**30
        eng = sgraph.Engine("pr", device_budget_gb=budget)
        try:
            eng.load_csr(row, col)
            eng.init()
            check(eng, row, col, f"budget {budget:.4f}")
            r, c = row, col
            for t in range(2):
                eng.apply(ins[t], dele[t])
                r, c = O.apply_updates(r, c, ins[t], dele[t])
                check(eng, r, c, f"budget {budget:.4f} G{t + 1}")
            whole[budget] = eng.values()
            assert eng.stats()["pull_rounds"] > 0
            if held is None:
                held = eng.stats()["device_bytes"]
            else:
                assert eng.stats()["device_bytes"] <= held - len(col)
        finally:
            eng.close()
    a, b = whole.values()
    assert float(np.max(np.abs(a.astype(np.float64) - b) / a)) <= 2 * PR_REL_TOL


def test_rounds_given_up_lose_no_mass():
    nv, row, col = sgraph.gen_rmat(11, 8, seed=97)
    ins, dele = sgraph.gen_updates(row, col, 11, 1, 500, 500, seed=98)
    full = sgraph.Engine("pr", pull_divisor=sgraph.PULL_ALWAYS)
    cut = sgraph.Engine("pr", pull_divisor=sgraph.PULL_ALWAYS, max_rounds=3)
    try:
        for e in (full, cut):
            e.load_csr(row, col)
        full.init()
        with pytest.raises(sgraph.SgError):
            cut.init()
        # ranks + what their residuals still have to deliver: r = value + M value' holds for
        # any push order, so the residual is exactly (1 - a) + a * M value - value
        v, res = cut.values().astype(np.float64), cut.gather(sgraph.Q_BUFFER).astype(np.float64)
        deg = np.maximum(np.diff(row.astype(np.int64)), 1)
        src = np.repeat(np.arange(nv), np.diff(row.astype(np.int64)))
        exp = 0.15 + 0.85 * np.bincount(col, weights=(v / deg)[src], minlength=nv) - v
        assert np.max(np.abs(res - exp)) <= 1e-5 * max(1.0, float(v.max()))
    finally:
        full.close()
        cut.close()
