"""Loads of engines with tiles of more particles than one workgroup holds
(8192), which are taken in pieces (GPU): every particle comes back whole, and
every slot of the storage holds one of the cell that the order by rank and cell
gives it (which one of a cell is open).  No arithmetic, no tolerance.
"""
from __future__ import annotations

import numpy as np
import pytest

import sputnipic_amd as S

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    yield


@pytest.mark.parametrize("order", ["load", "engine"])
@pytest.mark.parametrize("tile", [(4, 4, 4), (8, 4, 4)])
@pytest.mark.parametrize("spread", ["cell", "tile"])
@pytest.mark.parametrize("counts", [
    [8193, 3], [16384, 0, 8192], [5, 16385, 8193, 0, 9000], [100003, 1],
])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_pieces(counts, spread, tile, order, prec):
    r = np.random.default_rng(sum(counts))
    nx = 3 * tile[0] * len(counts)
    t = np.repeat(np.arange(len(counts)), counts)
    n = len(t)
    cit = [r.integers(0, m, n) if spread == "tile" else np.full(n, m - 1) for m in tile]
    # positions and charges that FP32 engines hold exactly
    p = {k: (c + (3 * t * tile[0] if k == "x" else 0) + r.integers(1, 256, n) / 256.0) * 0.5
         for k, c in zip("xyz", cit)}
    by = r.permutation(n)
    t, cit, p = t[by], [c[by] for c in cit], {k: v[by] for k, v in p.items()}
    for k in "uvw":
        p[k] = r.integers(-1000, 1000, n) / 256.0
    p["q"] = np.arange(n) + 1.0
    grd = S.Grid(nx, tile[1], tile[2], 0.5 * nx, 0.5 * tile[1], 0.5 * tile[2], prec)
    part = S.Particles(p, 1.0, "f64")
    eng = S.Engine(grd, 1, tile=tile,
                   order=S.SPIC_ORDER_ENGINE if order == "engine" else S.SPIC_ORDER_LOAD)
    try:
        for _ in range(2):  # the second into storage and workspace of the first
            for k, v in p.items():
                part.d[k].upload(v)
            eng.load(0, part)
            for k in p:
                part.d[k].upload(np.zeros(n))
            eng.store(0, part)
            got = part.download()
            at = np.asarray(got["q"]).astype(np.int64) - 1
            if order == "load":
                assert np.array_equal(at, np.arange(n))
            assert np.array_equal(np.sort(at), np.arange(n))
            for k in p:
                assert np.array_equal(got[k], p[k][at]), k
            if order == "engine":
                cell = (cit[0] * tile[1] + cit[1]) * tile[2] + cit[2]
                key = t * 1000 + cell
                by_key = np.argsort(key, kind="stable")
                first = np.searchsorted(key[by_key], key[by_key], side="left")
                rank = np.empty(n, np.int64)
                rank[by_key] = np.arange(n) - first
                want = np.lexsort((cell, rank, t))
                assert np.array_equal(key[at], key[want])
    finally:
        eng.close()
