"""The pull plan's packed tiles at every id width, on the CPU.

Ids of 1 to 32 bits, packed tile by tile by k_plan_ids: unpacked here, they are
the lists' ids again, the largest of each width among them. The pull kernels then
read tiles of every width (ids below the number of vertices): the sums they leave
are those of the lists. Edge counts around a tile, lists that cross tiles.
"""
import ctypes

import numpy as np
import pytest


TILE = 512  # kPullTile


def lists(r, nv, ne):
    """Lengths of nv lists, ne ids in all: many empty or short, one long."""
    deg = np.bincount(np.sort(r.integers(0, nv, ne) ** 2 // nv), minlength=nv)
    deg[nv // 2] += deg[0]
    deg[0] = 0
    return deg.astype(np.uint32)


def ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def plan(so, bits, deg, ids, push=None):
    nt = -(-len(ids) // TILE)
    words = np.zeros(nt * TILE // 32 * bits, np.uint32)
    sums = np.zeros(len(deg), np.float32)
    rc = so.emulation_pull_plan(ctypes.c_uint32(bits), ctypes.c_uint32(len(deg)), ptr(deg), ptr(ids), ctypes.c_uint64(len(ids)),
                                ptr(push) if push is not None else None, ptr(words), ptr(sums) if push is not None else None)
    assert rc == 0, "access out of bounds"
    return words, sums


def unpack(words, bits, n):
    b = np.unpackbits(words.view(np.uint8), bitorder="little").astype(np.uint64)
    at = (np.arange(n) // TILE) * (TILE * bits) + (np.arange(n) % TILE) * bits
    return sum(b[at + k] << np.uint64(k) for k in range(bits)).astype(np.uint32)


@pytest.mark.parametrize("bits", range(1, 33))
def test_ids_of_every_width(emulated, bits):
    r = np.random.default_rng(bits)
    for ne in (1, 511, 512, 513, 1500):
        ids = r.integers(0, 1 << bits, ne, dtype=np.uint64).astype(np.uint32)
        ids[::5] = (1 << bits) - 1
        words, _ = plan(emulated, bits, lists(r, 40, ne), ids)
        assert np.array_equal(unpack(words, bits, ne), ids)


@pytest.mark.parametrize("bits", [*range(8, 33, 3), 31])
def test_pulls_of_every_width(emulated, bits):
    r = np.random.default_rng(bits)
    nv = 256
    for ne in (1, 512, 513, 1700):
        deg = lists(r, nv, ne)
        ids = r.integers(0, nv, ne).astype(np.uint32)
        ids[::7] = nv - 1
        push = r.integers(1, 100, nv).astype(np.float32)  # sums stay exact
        _, sums = plan(emulated, bits, deg, ids, push)
        exp = np.bincount(np.repeat(np.arange(nv), deg), weights=push[ids], minlength=nv)
        assert np.array_equal(sums, exp)
