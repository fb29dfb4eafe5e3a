"""Results read through pinned staging: whole at the sizes where the chunks can go wrong.

Chunks of 512 KiB, eight to a launch, through sixteen staging slots: results just
below, at and above a chunk, a launch and the slots (and below the 512 KiB that
come in one piece), read twice into fresh memory.
Degrees are known without the device; OFFSETS are 8-byte words. Pointwise reads
of up to 65536 ids go through pinned words without copies.
"""
import numpy as np
import pytest

import sgraph

pytestmark = pytest.mark.gpu

MB = 1 << 18  # 4-byte words


@pytest.mark.parametrize("nv", [MB // 2 - 1, MB // 2, MB // 2 + 1, MB + 3, 4 * MB, 4 * MB + 1, 2 * MB - 1, 2 * MB, 2 * MB + 1, 3 * MB, 8 * MB + 1, 9 * MB - 3, 17 * MB + 5])
def test_results_come_whole(nv):
    rng = np.random.default_rng(nv)
    deg = rng.integers(0, 3, nv).astype(np.uint32)
    row = np.zeros(nv + 1, np.uint64)
    np.cumsum(deg, out=row[1:])
    u = np.repeat(np.arange(nv, dtype=np.int64), deg)
    k = np.arange(len(u)) - row[u].astype(np.int64)
    col = ((u + 1 + k) % nv).astype(np.uint32)
    eng = sgraph.Engine("cc")
    try:
        eng.load_csr(row, col)
        for _ in range(2):
            assert np.array_equal(eng.gather(sgraph.Q_DEGREE), deg)
        off = eng.gather(sgraph.Q_OFFSETS)
        assert off[-1] == eng.stats()["capacity"] and np.all(np.diff(off.astype(np.int64)) >= deg)
        eng.init()
        a = eng.values()
        b = eng.gather_at(np.arange(nv, dtype=np.uint32))
        assert np.array_equal(a, b)
    finally:
        eng.close()


@pytest.mark.parametrize("n", [1, 255, 257, 65535, 65536, 65537, 70001])
def test_lookups_at_the_end_of_the_pinned_words(n):
    nv = 3001
    rng = np.random.default_rng(n)
    u = rng.integers(0, nv - 1, 9000)
    k = np.unique(u * nv + u + 1)
    row = np.zeros(nv + 1, np.uint64)
    np.cumsum(np.bincount(k // nv, minlength=nv).astype(np.uint64), out=row[1:])
    eng = sgraph.Engine("cc")
    try:
        eng.load_csr(row, (k % nv).astype(np.uint32))
        eng.init()
        v = eng.values()
        ids = rng.integers(0, nv + 5, n).astype(np.uint32)  # ids past the graph read as 0xFFFFFFFF
        exp = np.where(ids < nv, v[np.minimum(ids, nv - 1)], 0xFFFFFFFF)
        assert np.array_equal(eng.gather_at(ids), exp)
        assert np.array_equal(eng.gather_at(ids[::-1]), exp[::-1])
    finally:
        eng.close()
