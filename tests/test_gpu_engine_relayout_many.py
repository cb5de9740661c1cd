"""Segments fitted anew on grids of more tiles than one workgroup lays out (GPU):
particles of a few tiles that move into the next ones and overflow them, then stay;
1023 to 2050 tiles, and 262500 (more than 1024 for each of 256 workgroups).  Every
particle is kept and the next layout holds them all; charges and positions to the
last bit (FP64; the step moves them by a whole number of units).
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("tiles", [(93, 11, 1), (128, 8, 1), (25, 41, 1), (41, 50, 1),
                                   (75, 70, 50)])
def test_layout(tiles, batch):
    S.set_async(False)
    S.set_strict_fp(False)
    cells = [4 * t for t in tiles]
    L = [0.5 * c for c in cells]
    grd = S.Grid(*cells, *L, "f64")
    r = np.random.default_rng(4)
    n, crowds = 20000, 12
    t = [r.integers(0, m, crowds) for m in tiles]
    t[0] = np.linspace(0, tiles[0] - 2, crowds).astype(np.int64)  # the last tiles too
    k = r.integers(0, crowds, n)
    # multiples of 1/64 inside the tile, so that a step of 2.0 is exact
    p = {c: 2.0 * t[a][k] + r.integers(7, 121, n) / 64.0 for a, c in enumerate("xyz")}
    dt = 0.25
    p["u"] = np.full(n, 2.0 / dt)
    p["v"] = p["w"] = np.zeros(n)
    p["q"] = r.uniform(0.5, 1.5, n)
    field = S.EMField(grd, {c: np.zeros(grd.nn) for c in O.FIELD_NAMES})
    part, ids = S.Particles(p, 1.0, "f64"), [S.InterpDensSpecies(grd)]
    param = S.Parameters(dt=dt, c=1.0, NiterMover=1)
    eng = S.Engine(grd, 1, set_moments=True)
    try:
        eng.load(0, part)
        if batch:
            many = S.Batch([(eng, field, ids, param)], set_moments=True)
            many.phase()
            many.close()
        else:
            eng.phase(field, ids, param)
        assert eng.stats()["overflow"] > 256
        for _ in range(2):  # deposits alone: the particles stay where they are
            eng.deposit(ids)
            assert eng.stats()["overflow"] == 0
        rho = ids[0].download()["rhon"]
        eng.store(0, part)
    finally:
        eng.close()
    got = part.download()
    for c in "yzq":
        assert np.array_equal(got[c], p[c]), c
    assert np.array_equal(got["x"], p["x"] + 2.0)
    total = float(np.sum(rho)) * 0.125
    assert abs(total - float(np.sum(p["q"]))) <= 1e-12 * n
