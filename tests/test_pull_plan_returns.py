"""A pull plan given back under a device budget returns when there is room again.

The caller's own device memory counts against the engine's budget: taking some
makes the engine give its plan back, and pulls read the store's slots. Once it
is freed, a later batch builds the plan anew; while it is held, none does.
"""
import numpy as np
import pytest

import oracle as O
import sgraph

PR_REL_TOL = 5e-5
NV, NE = 700, 20000


def test_plan_returns(backend):
    r = np.random.default_rng(41)
    k = r.permutation(NV * NV)[:NE + 200]
    first, fresh = np.sort(k[:NE]), np.stack([k // NV, k % NV], 1).astype(np.uint32)[NE:]
    row = np.zeros(NV + 1, np.uint64)
    np.cumsum(np.bincount(first // NV, minlength=NV), out=row[1:])
    col = (first % NV).astype(np.uint32)
    none = np.zeros((0, 2), np.uint32)
    ids = NE * 10 // 8  # 20,000 ids of 10 bits: the least a plan holds

    def stream(budget, taken):
        """Device bytes after the third batch, then after ten more with `taken` bytes
        held, then after ten with them free."""
        now = row, col
        eng = sgraph.Engine("pr", pull_divisor=sgraph.PULL_ALWAYS, device_budget_gb=budget / 2**30)
        held = []
        try:
            eng.load_csr(row, col)
            eng.init()
            p = None
            for t in range(23):
                if t == 3:
                    held.append(eng.stats()["device_bytes"])
                    p = eng.device_alloc(taken)
                if t == 13:
                    held.append(eng.stats()["device_bytes"] - taken)
                    eng.device_free(p)
                ins, dele = fresh[4 * t:4 * t + 4], none
                eng.apply(ins, dele)
                now = O.apply_updates(*now, ins, dele)
                if t in (2, 12, 22):
                    exp = O.pagerank(*now)
                    rel = np.max(np.abs(eng.values().astype(np.float64) - exp) / exp)
                    assert rel <= PR_REL_TOL, f"G{t + 1}: rel {rel}"
            held.append(eng.stats()["device_bytes"])
        finally:
            eng.close()
        return held

    room = stream(0, ids)
    held = stream(room[0] + ids // 2, ids)
    assert held[0] == room[0]
    assert held[1] + ids <= held[0], "the plan was not given back"
    assert held[2] >= held[0], "the plan did not return"
