"""The order in which a load puts a species' particles (GPU): tile by tile, each
tile round-robin over its cells (every cell's first particle, then every
cell's second, ...), the particles of a cell in the caller's order.  It decides
in which order an engine sums, which in FP32 shows.  An engine without load index
stores in its own order, so the stored charges show it; no tolerance.
"""
from __future__ import annotations

import numpy as np
import pytest

import sputnipic_amd as S

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield


def _expected(cells, tile, pos, d):
    """Caller indices in storage order."""
    c = [np.minimum((p / d).astype(np.int64), m - 1) for p, m in zip(pos, cells)]
    nt = [-(-m // t) for m, t in zip(cells, tile)]
    t = [a // b for a, b in zip(c, tile)]
    r = [a % b for a, b in zip(c, tile)]
    tid = (t[0] * nt[1] + t[1]) * nt[2] + t[2]
    cit = (r[0] * tile[1] + r[1]) * tile[2] + r[2]
    cell = tid * (tile[0] * tile[1] * tile[2]) + cit
    by_cell = np.argsort(cell, kind="stable")
    start = np.searchsorted(cell[by_cell], cell[by_cell], side="left")
    rank = np.empty(len(cell), np.int64)
    rank[by_cell] = np.arange(len(cell)) - start
    return np.lexsort((cit, rank, tid))


CASES = [
    ((4, 4, 4), 1, "random"),
    ((8, 4, 4), 8191, "random"), ((4, 4, 4), 8192, "random"),
    ((1, 4, 4), 8192, "random"),        # 512 particles in each of 16 cells
    ((1, 1, 4), 1023, "random"),        # 256 in each of four
    ((13, 9, 6), 5003, "random"),
    ((64, 40, 40), 300001, "random"),   # a few particles per cell
    ((16, 16, 16), 131072, "random"),
    # as many per cell, cell by cell (a cell's particles in one wave)
    ((13, 9, 6), 2, "cells"), ((13, 9, 6), 8, "cells"), ((5, 4, 4), 64, "cells"),
    ((16, 16, 16), 32, "cells"), ((40, 32, 30), 1, "cells"),
    # 2197 tiles of 64 particles, and of fewer
    ((52, 52, 52), 1, "cells"), ((52, 52, 51), 1, "cells"),
]


@pytest.mark.parametrize("prec,src", [("f64", "f64"), ("f32", "f32"), ("f32", "f64")])
@pytest.mark.parametrize("tile", [(4, 4, 4), (8, 4, 4)])
@pytest.mark.parametrize("cells,n,order", CASES)
def test_order_of_a_load(cells, n, order, tile, prec, src):
    per_tile = tile[0] * tile[1] * tile[2]
    tiles = np.prod([-(-c // t) for c, t in zip(cells, tile)])
    if prec == "f32" and order == "random" and n < 4 * per_tile * tiles:
        pytest.skip("few FP32 particles: a cell's come wave by wave")
    d = 0.5
    dt = {"f64": np.float64, "f32": np.float32}[src]
    r = np.random.default_rng(n)
    if order == "cells":
        per, n = n, n * cells[0] * cells[1] * cells[2]
        c = np.arange(n) // per
        c = [c // (cells[1] * cells[2]), c // cells[2] % cells[1], c % cells[2]]
    else:
        c = [r.integers(0, m, n) for m in cells]
        if cells[0] == 1:  # as many in every cell
            c[1], c[2] = np.divmod(r.permutation(np.arange(n) % (cells[1] * cells[2])), cells[2])
    # positions that both precisions hold exactly and that lie inside cells
    pos = [(a + r.integers(1, 256, n) / 256.0) * d for a in c]
    p = {k: v.astype(dt) for k, v in zip("xyz", pos)}
    for k in "uvw":
        p[k] = np.zeros(n, dt)
    p["q"] = (1.0 + np.arange(n)).astype(dt)  # the caller's index, exact in FP32
    grd = S.Grid(*cells, d * cells[0], d * cells[1], d * cells[2], prec)
    part = S.Particles(p, 1.0, src)
    eng = S.Engine(grd, 1, tile=tile, order=S.SPIC_ORDER_ENGINE)
    want = _expected(cells, tile, pos, d)
    try:
        for _ in range(2):
            part.d["q"].upload(p["q"])
            for k, v in zip("xyz", pos):
                part.d[k].upload(v.astype(dt))
            eng.load(0, part)
            eng.store(0, part)
            got = np.asarray(part.download()["q"])
            assert np.array_equal(got, p["q"][want])
    finally:
        eng.close()
