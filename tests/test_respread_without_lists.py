"""Re-spread windows that hold a source with deletes but no list and no inserts.

Such a source has nothing to filter (no chunk of its own), and nothing of it
may be placed: neither the chunk of the next source with deletes nor what an
earlier, larger batch left past the end of the chunk list is its own. Full
stores (density 1.0), so that any insert past a source's range re-spreads.
"""
import numpy as np
import pytest

import oracle as O
import sgraph


def csr(lists, nv):
    row = np.zeros(nv + 1, np.uint64)
    np.cumsum([len(lists.get(v, ())) for v in range(nv)], out=row[1:])
    return row, np.concatenate([np.asarray(lists[v], np.uint32) for v in sorted(lists)])


def pairs(p):
    return np.array(p, np.uint32).reshape(-1, 2)


def check(eng, row, col):
    r, c = eng.adjacency()[:2]
    assert np.array_equal(np.asarray(r, np.uint64), row)
    assert np.array_equal(c, col), f"first at entry {int(np.argmax(c != col))}"


def test_stale_chunk_past_the_list(backend):
    # three hubs updated in place leave three chunk entries; in a smaller batch one
    # hub is updated and a list grows (two chunks), and the last vertex, which has no
    # list, comes after them (the
    # lists fill the store: every vertex is moved)
    nv = 1100
    row, col = csr({**{v: range(10, 1010) for v in range(7)}, 8: [1, 2, 3]}, nv)
    eng = sgraph.Engine("bfs", pma_density=1.0, round_blocks=8)
    try:
        eng.load_csr(row, col)
        eng.init(3)
        for ins, dele in (([], [(3, 11)] * 1200 + [(4, 21), (5, 31)]), ([(8, 50 + k) for k in range(1000)], [(3, 12), (nv - 1, 7)])):
            eng.apply(pairs(ins), pairs(dele))
            row, col = O.apply_updates(row, col, pairs(ins), pairs(dele))
            check(eng, row, col)
        assert eng.stats()["resizes"] == 1
        assert np.array_equal(eng.values(), O.bfs(row, col, 3))
    finally:
        eng.close()


@pytest.mark.parametrize("nq", [0, 17, 70])
def test_neighbours_keep_their_lists(backend, nq):
    # every fourth vertex is empty and has an absent edge deleted, next to a list
    # of 30 that loses one; one list outgrows its range
    if backend is not None:
        backend.emulation_backwards()  # an empty source comes after its neighbours
    nv = 600
    row, col = csr({v: (v + 1 + np.arange(30)) % nv for v in range(nv) if v % 4 != 3}, nv)
    dele = pairs([(v, 5) if v % 4 == 3 else (v, (v + 9) % nv) for v in range(nv) if v % 4 in (0, 3)])
    ins = pairs([(1, 100 + k) for k in range(200)])
    eng = sgraph.Engine("multi" if nq else "cc", weight_mode="seeded", weight_seed=7, pma_density=1.0, round_blocks=8)
    try:
        eng.load_csr(row, col)
        sources = (np.arange(nq) * 8 % nv).astype(np.uint32)
        if nq:
            eng.init_queries(sources, ["sssp"] * nq)
        else:
            eng.init()
        for i, d in ((ins, dele), (dele[:20], ins[::2])):
            eng.apply(i, d)
            row, col = O.apply_updates(row, col, i, d)
            check(eng, row, col)
        assert eng.stats()["rebalances"] > 0
        if not nq:
            assert np.array_equal(eng.values(), O.cc(row, col))
        for q in range(nq):
            assert np.array_equal(eng.query(q), O.sssp(row, col, int(sources[q]), "seeded", 7)), f"query {q}"
    finally:
        eng.close()
