"""The caller-order deposit through tiles (interpP2G and mover_interp of
enough particles) against the oracle: counts around the threshold and the
staged batches, every particle in one cell (several work items of one tile),
grids whose last tile is partial, any particle order, the upper faces (ghost
cells), particles outside the grid, and a captured call (the direct kernels).

Tolerances: particle state bit for bit in strict arithmetic; moments, whose
terms are the oracle's summed in another order in FP64, within 1e-13 of each
array's maximum (FP64) and 1e-5 of the FP32 oracle, which sums in float.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_bitwise, assert_close

pytestmark = pytest.mark.gpu

# 9 x 6 x 5 cells: 3 x 2 x 2 tiles over the deposit cells, the last ones partial
CFG = dict(nxc=9, nyc=6, nzc=5, Lx=4.5, Ly=3.0, Lz=2.5, npcelx=[1] * 4, npcely=[1] * 4,
           npcelz=[1] * 4, B0x=0.2, uth=[0.05] * 4, vth=[0.05] * 4, wth=[0.05] * 4)


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield
    S.set_async(False)
    S.set_strict_fp(False)


def _particles(cfg, n, kind, prec, seed=3):
    r = np.random.default_rng(seed)
    dt = np.float64 if prec == "f64" else np.float32
    box = (cfg.Lx, cfg.Ly, cfg.Lz)
    p = {}
    for a, L in zip("xyz", box):
        x = r.uniform(0.0, 1.0, n)
        if kind == "one_cell":
            x = 0.5 + (x - 0.5) * 0.05
        p[a] = (x * L * (1 - 1e-6)).astype(dt)
    if kind == "faces":  # on the upper faces: the deposit cell is a ghost cell
        p["x"][::3] = dt(cfg.Lx)
        p["y"][::5] = dt(cfg.Ly)
        p["z"][::7] = dt(cfg.Lz)
    for a in "uvw":
        p[a] = r.normal(0.0, 0.05, n).astype(dt)
    p["q"] = r.uniform(0.5, 1.5, n).astype(dt)
    if kind == "sorted":
        order = np.lexsort([np.floor(p[a] * 2) for a in "zyx"])
        p = {k: v[order] for k, v in p.items()}
    return p


def _pair(n, kind, prec):
    cfg = O.GemConfig(**CFG)
    st = O.State(cfg, prec)
    st.parts = [_particles(cfg, n, kind, prec)]
    dt = np.float64 if prec == "f64" else np.float32
    grd = S.Grid(cfg.nxc, cfg.nyc, cfg.nzc, cfg.Lx, cfg.Ly, cfg.Lz, prec)
    field = S.EMField(grd, {k: st.fields[k].astype(dt) for k in O.FIELD_NAMES})
    part = S.Particles(st.parts[0], cfg.qom[0], prec, cfg.NiterMover)
    param = S.Parameters(dt=cfg.dt, c=cfg.c, NiterMover=cfg.NiterMover)
    return cfg, st, grd, field, part, S.InterpDensSpecies(grd), param


@pytest.mark.parametrize("strict", [True, False])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,kind", [(12287, "uniform"), (12288, "uniform"), (12289, "sorted"),
                                    (25 * 512, "one_cell"), (25 * 512 + 1, "one_cell"),
                                    (30011, "uniform"), (30011, "sorted"), (15000, "faces")])
def test_deposit_matches_oracle(n, kind, prec, strict):
    _, st, grd, _, part, ids, _ = _pair(n, kind, prec)
    S.set_strict_fp(strict)
    S.interpP2G(part, ids, grd)
    st.zero_moments(0)
    st.interp_p2g(0)
    m = ids.download()
    for k in O.MOMENT_NAMES:
        assert_close(m[k], st.moments[0][k], 1e-13 if prec == "f64" else 1e-5, k)


@pytest.mark.parametrize("grid", [(88, 72, 64), (97, 49, 41)])
def test_many_tiles(grid):
    """More tiles than a workgroup counts in LDS, and fewer; total charge and
    the oracle's moments."""
    n = 60000
    cfg = O.GemConfig(**dict(CFG, nxc=grid[0], nyc=grid[1], nzc=grid[2]))
    st = O.State(cfg, "f64", build_ic=False)
    st.parts = [_particles(cfg, n, "uniform", "f64")]
    grd = S.Grid(*grid, cfg.Lx, cfg.Ly, cfg.Lz, "f64")
    part, ids = S.Particles(st.parts[0], 1.0, "f64"), S.InterpDensSpecies(grd)
    S.interpP2G(part, ids, grd)
    st.zero_moments(0)
    st.interp_p2g(0)
    m = ids.download()
    for k in O.MOMENT_NAMES:
        assert_close(m[k], st.moments[0][k], 1e-13, k)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,kind", [(12288, "sorted"), (30011, "uniform"), (12801, "one_cell")])
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


def test_particle_outside_the_grid_is_reported():
    cfg, _, grd, _, part, ids, _ = _pair(16000, "uniform", "f64")
    p = part.download()
    p["y"][4321] = -3 * cfg.Ly / cfg.nyc
    with pytest.raises(S.SpicError) as ei:
        S.interpP2G(S.Particles(p, 1.0, "f64"), ids, grd)
    assert ei.value.code == S.SPIC_EDOMAIN
    S.interpP2G(part, ids, grd)  # the flag does not stay


def test_captured_deposit_replays():
    """A captured call cannot allocate and takes the direct kernels."""
    from sputnipic_amd import core
    _, st, grd, _, part, ids, _ = _pair(16384, "uniform", "f64")
    st.zero_moments(0)
    st.interp_p2g(0)
    s = S.Stream()
    g, sp, m = grd.c_struct(), part.c_struct(), ids.c_struct()
    with S.Graph(s) as graph:
        core.check(core.lib().spic_zero_moments(core.C.byref(g), core.C.byref(m), s.ptr), "zero")
        core.check(core.lib().spic_interp_p2g(core.C.byref(g), core.C.byref(sp), core.C.byref(m),
                                              s.ptr), "interp")
    for _ in range(3):
        graph.launch()
        s.synchronize()
        got = ids.download()
        for k in O.MOMENT_NAMES:
            assert_close(got[k], st.moments[0][k], 1e-13, k)
    graph.close()
