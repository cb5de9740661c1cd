"""Caller-order deposits at the limits of the way through tiles (16384 particles,
and eight per tile, on) and of the forms it takes: one particle less and more,
several work items of one tile, upper faces (ghost cells), particles outside the
grid, counters in LDS with several particles per thread, places of 4096 particles,
work items of several batches, and up to 6144 tiles and more.

Tolerances as for the smaller counts: particle state bit for bit in strict
arithmetic; moments within 1e-13 of each array's maximum (FP64, the oracle's terms
in another order; 1e-12 for a million) and 1e-5 of the FP32 oracle, which sums in
float.  Where it sums a hundred thousand FP32 particles per node, the FP64 oracle's
sums of the same particles take its place: ten roundings of a term, 10 * 2^-24 =
6e-7, rounded up to 1e-6 (node coordinates are multiples of 0.5, alike in both).
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_bitwise, assert_close
from test_gpu_deposit_tiles import CFG, _pair, _particles

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield
    S.set_async(False)
    S.set_strict_fp(False)


COUNTS = [(16383, "uniform"), (16384, "uniform"), (16385, "sorted"), (33 * 512, "one_cell"),
          (33 * 512 + 1, "one_cell"), (16385, "faces"), (20011, "faces")]


@pytest.mark.parametrize("strict", [True, False])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,kind", COUNTS)
def test_deposit_matches_oracle(n, kind, prec, strict):
    _, st, grd, _, part, ids, _ = _pair(n, kind, prec)
    S.set_strict_fp(strict)
    S.interpP2G(part, ids, grd)
    st.zero_moments(0)
    st.interp_p2g(0)
    m = ids.download()
    for k in O.MOMENT_NAMES:
        assert_close(m[k], st.moments[0][k], 1e-13 if prec == "f64" else 1e-5, k)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,kind", [c for c in COUNTS if c[1] != "faces"])
def test_fused_matches_oracle(n, kind, prec):
    _, st, grd, field, part, ids, param = _pair(n, kind, prec)
    S.set_strict_fp(True)
    S.mover_interp(part, field, ids, grd, param)
    st.zero_moments(0)
    st.mover_interp(0)
    got, m = part.download(), ids.download()
    for k in O.PARTICLE_NAMES:
        assert_bitwise(got[k], st.parts[0][k], k)
    for k in O.MOMENT_NAMES:
        assert_close(m[k], st.moments[0][k], 1e-13 if prec == "f64" else 1e-5, k)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("axis,side", [("x", 1), ("y", -1), ("z", 1)])
def test_particle_outside_the_grid_is_reported(axis, side, fused, prec):
    cfg, _, grd, field, part, ids, param = _pair(20000, "uniform", prec)
    p = part.download()
    L = {"x": cfg.Lx, "y": cfg.Ly, "z": cfg.Lz}[axis]
    p[axis][4321] = -L if side < 0 else 2 * L
    bad = S.Particles(p, 1.0, prec)
    with pytest.raises(S.SpicError) as ei:
        if fused:
            S.mover_interp(bad, field, ids, grd, param)
        else:
            S.interpP2G(bad, ids, grd)
    assert ei.value.code == S.SPIC_EDOMAIN
    S.interpP2G(part, ids, grd)  # the flag does not stay


def _big(grid, n, kind, prec, fused=False):
    """Deposit of n particles against the oracle's, in FP64 on the coarse grid."""
    ref = "f64" if grid == (9, 6, 5) else prec
    rel = 1e-12 if prec == "f64" else 1e-6 if ref == "f64" else 1e-5
    cfg = O.GemConfig(**dict(CFG, nxc=grid[0], nyc=grid[1], nzc=grid[2]))
    p = _particles(cfg, n, kind, prec)
    grd = S.Grid(*grid, cfg.Lx, cfg.Ly, cfg.Lz, prec)
    part, ids = S.Particles(p, 1.0, prec), S.InterpDensSpecies(grd)
    if fused:
        S.mover_interp(part, S.EMField(grd), ids, grd, S.Parameters(dt=1e-3, c=1.0))
        p = part.download()
    else:
        S.interpP2G(part, ids, grd)
    st = O.State(cfg, ref, build_ic=False)
    st.parts = [{k: np.asarray(v).astype(np.float64 if ref == "f64" else np.float32)
                 for k, v in p.items()}]
    st.zero_moments(0)
    st.interp_p2g(0)
    m = ids.download()
    for k in O.MOMENT_NAMES:
        assert_close(m[k], st.moments[0][k], rel, k)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("grid,n,kind", [
    ((9, 6, 5), 1100003, "uniform"),     # two particles per thread counted, places of 4096
    ((9, 6, 5), 1100003, "one_cell"),    # work items of 1024 and more, all of one tile
    ((40, 40, 40), 600001, "sorted"),    # places of 4096, one per thread counted
    ((53, 51, 50), 1100003, "uniform"),  # 2366 tiles
    ((76, 72, 66), 1100003, "uniform"),  # 6460 tiles: more than the LDS counters
])
def test_many_particles(grid, n, kind, prec):
    _big(grid, n, kind, prec)
