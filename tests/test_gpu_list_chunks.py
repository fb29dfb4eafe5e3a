"""Batch updates of lists around the merge chunk (2048 entries) and the wave.

One list of exactly n entries, n around one chunk, two, and 64 chunks (more
than a wave's lanes), takes deletes at its ends and at the chunk boundaries and
inserts around the 128 that one lane appends; once with room (updated in place
or through staging) and once in a full store (moved by a re-spread). The lists
are compared with the oracle's, entry by entry.
"""
import numpy as np
import pytest

import oracle as O
import sgraph

pytestmark = pytest.mark.gpu

CHUNK = 2048


@pytest.mark.parametrize("density", [0.25, 1.0])
@pytest.mark.parametrize("n", [1, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK, 64 * CHUNK, 64 * CHUNK + 1, 65 * CHUNK + 7])
@pytest.mark.parametrize("nins", [0, 1, 128, 129, CHUNK + 1])
def test_list_around_the_chunks(n, nins, density):
    nv = 160000
    hub, other = 7, 11
    row = np.zeros(nv + 1, np.uint64)
    deg = np.zeros(nv, np.int64)
    deg[hub], deg[other], deg[other + 1:other + 50] = n, 300, 3
    np.cumsum(deg, out=row[1:])
    col = np.concatenate([np.arange(n) + 20, np.arange(300) + 1000, np.tile([5, 6, 7], 49)]).astype(np.uint32)
    at = sorted({0, n // 2, n - 1, *(k for k in range(CHUNK - 1, n, CHUNK)), *(k for k in range(CHUNK, n, CHUNK))})
    dele = np.array([(hub, 20 + k) for k in at] + [(other + 3, 6), (other + 3, 9)], dtype=np.uint32)
    ins = np.array([(hub, 20 + n + k) for k in range(nins)] + [(other, 5000 + k) for k in range(nins)],
                   dtype=np.uint32).reshape(-1, 2)
    eng = sgraph.Engine("bfs", pma_density=density)
    try:
        eng.load_csr(row, col)
        eng.init(hub)
        r, c = row, col
        for i, d in ((ins, dele), (dele[:-1], ins[: nins // 2])):
            eng.apply(i, d)
            r, c = O.apply_updates(r, c, i, d)
            gr, gc = eng.adjacency()[:2]
            assert np.array_equal(gr.astype(np.uint64), np.asarray(r, np.uint64)) and np.array_equal(gc, c)
        assert np.array_equal(eng.values(), O.bfs(r, c, hub))
    finally:
        eng.close()
