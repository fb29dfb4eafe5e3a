"""Entries that are no vertex, planted in live lists of the emulated engine.

Updates leave none there; batched walks, which index their state with what they
read, skip one all the same.
"""
import numpy as np
import pytest

import oracle as O
import sgraph

GAP = 0xFFFFFFFF


def graph():
    """600 vertices; target 599 stands in 9 lists: short ones, one of 70 and one of 700."""
    nv = 600
    lists = {v: [(v * 5 + k) % 590 for k in range(1 + v % 9)] for v in range(0, 590, 3)}
    lists[1] = [(3 + k) % 590 for k in range(69)]
    lists[2] = [(k * 7) % 590 for k in range(699)]
    for v in (0, 3, 9, 42, 300, 501, 585):
        lists[v] = lists[v][:2] + [599] + lists[v][2:]
    lists[1].insert(66, 599)
    lists[2].insert(650, 599)
    row = np.zeros(nv + 1, np.uint64)
    np.cumsum([len(lists.get(v, ())) for v in range(nv)], out=row[1:])
    col = np.concatenate([np.asarray(lists[v], np.uint32) for v in sorted(lists)])
    return nv, row, col


@pytest.mark.parametrize("nq", [3, 17, 40, 70])
def test_batched_walks(emulated, nq):
    nv, row, col = graph()
    sources = (np.arange(nq) * 13 % 590).astype(np.uint32)
    sources[:3] = (0, 1, 2)
    eng = sgraph.Engine("multi", weight_mode="seeded", weight_seed=7, round_blocks=8)
    try:
        eng.load_csr(row, col)
        assert emulated.emulation_replace(599, GAP) >= 9
        eng.init_queries(sources, ["bfs", "sssp"] * (nq // 2) + ["bfs"] * (nq % 2))
        # the same with the entries gone
        src = np.repeat(np.arange(nv, dtype=np.uint32), np.diff(row.astype(np.int64)))
        r, c = O.apply_updates(row, col, np.zeros((0, 2), np.uint32), np.stack([src, col], 1)[col == 599])
        # resets walk the lists as well
        dele = np.stack([src, col], 1)[(col != 599)][::7]
        for t in range(2):
            for q in range(nq):
                s = int(sources[q])
                exp = O.sssp(r, c, s, "seeded", 7) if q % 2 else O.bfs(r, c, s)
                assert np.array_equal(eng.query(q), exp), f"G{t} query {q}"
            if t == 0:
                eng.apply(np.zeros((0, 2), np.uint32), dele)
                r, c = O.apply_updates(r, c, np.zeros((0, 2), np.uint32), dele)
    finally:
        eng.close()
