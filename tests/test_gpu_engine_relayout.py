"""Segments fitted anew when an overflow region has filled (GPU): a species
whose particles move from one tile into another, far more than the segment's
free slots, so that a phase leaves hundreds in the overflow region; the next
phase's segments hold them all.  Counts on both sides of the threshold of 256
overflow particles, an engine and a batch, FP64 and fixed-point FP32, and the
list ring's edges (all particles of a batch leave their tile).

Free streaming (no field): positions against the exact ones, charge
conserved, and the moments against the oracle's deposit of the same particles
(1e-13 of each array's maximum in FP64; 1e-5 in FP32).
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_close

pytestmark = pytest.mark.gpu

CFG = dict(nxc=12, nyc=4, nzc=4, Lx=6.0, Ly=2.0, Lz=2.0, npcelx=[1] * 4, npcely=[1] * 4,
           npcelz=[1] * 4)
SLACK = 16


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield


def _crowd(n, prec):
    """n particles of the first of three tiles that move one tile per step."""
    cfg = O.GemConfig(**CFG)
    r = np.random.default_rng(11)
    dt = np.float64 if prec == "f64" else np.float32
    dx = cfg.Lx / cfg.nxc
    p = {"x": r.uniform(0.1, 1.9, n), "y": r.uniform(0.1, 1.9, n), "z": r.uniform(0.1, 1.9, n)}
    p["u"] = np.full(n, 4 * dx / cfg.dt)
    for k in "vw":
        p[k] = np.zeros(n)
    p["q"] = r.uniform(0.5, 1.5, n)
    return cfg, {k: v.astype(dt) for k, v in p.items()}


def _run(n, prec, phases, batch):
    cfg, p = _crowd(n, prec)
    grd = S.Grid(cfg.nxc, cfg.nyc, cfg.nzc, cfg.Lx, cfg.Ly, cfg.Lz, prec)
    zero = np.zeros(grd.nn, np.float64 if prec == "f64" else np.float32)
    field = S.EMField(grd, {k: zero for k in O.FIELD_NAMES})
    param = S.Parameters(dt=cfg.dt, c=cfg.c, NiterMover=3)
    part, ids = S.Particles(p, 1.0, prec), [S.InterpDensSpecies(grd)]
    eng = S.Engine(grd, 1, set_moments=True, positions=0)
    overflow = []
    try:
        eng.load(0, part)
        many = S.Batch([(eng, field, ids, param)], set_moments=True) if batch else None
        for _ in range(phases):
            many.phase() if batch else eng.phase(field, ids, param)
            overflow.append(eng.stats()["overflow"])
        eng.store(0, part)
        got, mom = part.download(), ids[0].download()
        if many:
            many.close()
    finally:
        eng.close()
    return cfg, p, got, mom, overflow


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 129, 256, 257, 290, 1000, 9001])
def test_crowd_moves_on(n, prec, batch):
    phases = 2  # a third would carry iterates out of the grid
    cfg, p, got, mom, overflow = _run(n, prec, phases, batch)
    x = (p["x"].astype(np.float64) + phases * 2.0) % cfg.Lx
    d = np.abs(got["x"].astype(np.float64) - x)
    d = np.minimum(d, cfg.Lx - d)
    assert np.max(d) <= (1e-12 if prec == "f64" else 1e-5)
    for k in ("y", "z", "q"):
        assert np.max(np.abs(got[k] - p[k])) <= (0.0 if prec == "f64" else 3e-7)
    # a third of the mean holds 12% of slack; the rest of the crowd overflows
    assert (overflow[0] > 0) == (n > 3 * SLACK)
    st = O.State(cfg, prec, build_ic=False)
    st.parts = [got]
    st.zero_moments(0)
    st.interp_p2g(0)
    for k in O.MOMENT_NAMES:
        assert_close(mom[k], st.moments[0][k], 1e-13 if prec == "f64" else 1e-5, k)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_a_full_overflow_region_empties(prec):
    """Particles at rest after the first step: the second phase's segments hold
    every one of them."""
    cfg, p = _crowd(3000, prec)
    grd = S.Grid(cfg.nxc, cfg.nyc, cfg.nzc, cfg.Lx, cfg.Ly, cfg.Lz, prec)
    zero = np.zeros(grd.nn, np.float64 if prec == "f64" else np.float32)
    field = S.EMField(grd, {k: zero for k in O.FIELD_NAMES})
    part, ids = S.Particles(p, 1.0, prec), [S.InterpDensSpecies(grd)]
    eng = S.Engine(grd, 1, set_moments=True)
    try:
        eng.load(0, part)
        eng.phase(field, ids, S.Parameters(dt=cfg.dt, c=cfg.c))
        assert eng.stats()["overflow"] > 256
        # deposits alone: the particles stay where they are
        eng.deposit(ids)
        assert eng.stats()["overflow"] == 0
        eng.store(0, part)
    finally:
        eng.close()
    got = part.download()
    assert abs(float(np.sum(got["q"])) - float(np.sum(p["q"]))) <= 1e-6 * 3000
