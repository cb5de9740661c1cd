"""Species of a tile in workgroups side by side or in turn (GPU): grids of
few tiles, and of 255 and 256 tiles, on both sides of the line between the
two, against one engine per species and against the oracle's deposit.

Positions and velocities do not depend on the split: equal to the last bit.
Moments of the same particles add up in another order: 1e-13 of each array's
maximum in FP64; 1e-5 in FP32 against the oracle.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_close

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield


def _species(cfg, prec, counts):
    r = np.random.default_rng(5)
    dt = np.float64 if prec == "f64" else np.float32
    out = []
    for n in counts:
        p = {"x": r.uniform(0, 0.999 * cfg.Lx, n), "y": r.uniform(0.1, 0.9 * cfg.Ly, n),
             "z": r.uniform(0, 0.999 * cfg.Lz, n), "q": r.uniform(0.5, 1.5, n)}
        for k in "uvw":
            p[k] = r.normal(0, 0.02, n)
        out.append({k: v.astype(dt) for k, v in p.items()})
    return out


def _run(grd, field, param, parts, prec, push):
    ns = len(parts)
    P = [S.Particles(p, -1.0 + 2 * s, prec) for s, p in enumerate(parts)]
    ids = [S.InterpDensSpecies(grd) for _ in parts]
    eng = S.Engine(grd, ns, set_moments=True)
    try:
        for s in range(ns):
            eng.load(s, P[s])
        for _ in range(2):
            eng.phase(field, ids, param) if push else eng.deposit(ids)
        for s in range(ns):
            eng.store(s, P[s])
    finally:
        eng.close()
    return [p.download() for p in P], [i.download() for i in ids]


@pytest.mark.parametrize("push", [True, False])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("cells", [(5, 4, 4), (68, 20, 12), (64, 16, 16)])
@pytest.mark.parametrize("counts", [(4000, 0, 700), (1, 3000)])
def test_split_matches_one_species(cells, counts, prec, push):
    nx, ny, nz = cells
    cfg = O.GemConfig(nxc=nx, nyc=ny, nzc=nz, Lx=0.5 * nx, Ly=0.5 * ny, Lz=0.5 * nz,
                      npcelx=[1] * 4, npcely=[1] * 4, npcelz=[1] * 4)
    grd = S.Grid(cfg.nxc, cfg.nyc, cfg.nzc, cfg.Lx, cfg.Ly, cfg.Lz, prec)
    r = np.random.default_rng(6)
    dt = np.float64 if prec == "f64" else np.float32
    field = S.EMField(grd, {k: r.normal(0, 0.01, grd.nn).astype(dt) for k in O.FIELD_NAMES})
    param = S.Parameters(dt=cfg.dt, c=cfg.c, NiterMover=3)
    parts = _species(cfg, prec, counts)
    got, mom = _run(grd, field, param, parts, prec, push)
    for s, p in enumerate(parts):
        if not counts[s]:
            assert all(not np.any(mom[s][k]) for k in O.MOMENT_NAMES)
            continue
        P, ids = S.Particles(p, -1.0 + 2 * s, prec), S.InterpDensSpecies(grd)
        eng = S.Engine(grd, 1, set_moments=True)
        try:
            eng.load(0, P)
            for _ in range(2):
                eng.phase(field, [ids], param) if push else eng.deposit([ids])
            eng.store(0, P)
        finally:
            eng.close()
        one = P.download()
        for k in "xyzuvwq":
            assert np.array_equal(got[s][k], one[k]), k
        st = O.State(cfg, prec, build_ic=False)
        st.parts = [got[s]]
        st.zero_moments(0)
        st.interp_p2g(0)
        for k in O.MOMENT_NAMES:
            assert_close(mom[s][k], st.moments[0][k], 1e-13 if prec == "f64" else 1e-5, k)
