"""Loads through tiles and stores by line (GPU): particles per tile and per
cell at the edges of what a workgroup holds, both ways of counting and placing
(few and many tiles), every precision pair, against the caller's own arrays
and the oracle's deposit.

A load and a store move values: FP64 and FP32 velocities and charges come back
to the last bit, positions of an FP32 engine within the spacing of float
numbers at the box's end (4e-6 at 40) and the fixed-point unit: 1e-5.  The
order in a tile shows in the deposit of what was loaded: 1e-13 of each array's
maximum in FP64; in FP32 that spacing over a cell of 0.5, on three axes, in
sums that may cancel: 5e-5.
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


def _cfg(cells):
    nx, ny, nz = cells
    return O.GemConfig(nxc=nx, nyc=ny, nzc=nz, Lx=0.5 * nx, Ly=0.5 * ny, Lz=0.5 * nz,
                       npcelx=[1] * 4, npcely=[1] * 4, npcelz=[1] * 4)


def _check(cfg, p, prec, src, ids=True):
    """Load p (element type src) into an engine of precision prec, deposit,
    store, compare."""
    dt = {"f64": np.float64, "f32": np.float32}
    p = {k: v.astype(dt[src]) for k, v in p.items()}
    n = len(p["x"])
    grd = S.Grid(cfg.nxc, cfg.nyc, cfg.nzc, cfg.Lx, cfg.Ly, cfg.Lz, prec)
    part, mom = S.Particles(p, 1.0, src), [S.InterpDensSpecies(grd)]
    eng = S.Engine(grd, 1, set_moments=True, order=0 if ids else S.SPIC_ORDER_ENGINE)
    try:
        for _ in range(2):  # the second on storage and workspace kept from the first
            eng.load(0, part)
        assert eng.stats()["overflow"] == 0
        eng.deposit(mom)
        for k in "xyzuvwq":
            part.d[k].upload(np.zeros(n, dt[src]))
        eng.store(0, part)
    finally:
        eng.close()
    got, mom = part.download(), mom[0].download()
    if not ids:  # storage order: the same particles, by their charge
        assert len(np.unique(p["q"])) == n
        a, b = np.argsort(got["q"]), np.argsort(p["q"])
        got = {k: v[a] for k, v in got.items()}
        p = {k: v[b] for k, v in p.items()}
    for k in "xyz":
        if prec == "f64":
            assert np.array_equal(got[k], p[k]), k
        else:
            assert np.all(np.abs(got[k].astype(np.float64) - p[k]) <= 1e-5), k
    for k in "uvwq":
        want = p[k] if prec == "f64" else p[k].astype(np.float32).astype(dt[src])
        assert np.array_equal(got[k], want), k
    st = O.State(cfg, prec, build_ic=False)
    st.parts = [{k: v.astype(dt[prec]) for k, v in got.items()}]
    st.zero_moments(0)
    st.interp_p2g(0)
    for k in O.MOMENT_NAMES:
        assert_close(mom[k], st.moments[0][k], 1e-13 if prec == "f64" else 5e-5, k)


def _fill(n, r, q0=0.5):
    p = {k: r.normal(0, 0.1, n) for k in "uvw"}
    p["q"] = r.permutation(np.linspace(q0, q0 + 1, n, endpoint=False)) if n else np.zeros(0)
    return p


PAIRS = [("f64", "f64"), ("f32", "f32"), ("f32", "f64")]


@pytest.mark.parametrize("prec,src", PAIRS)
@pytest.mark.parametrize("n", [1, 511, 512, 513, 4095, 4096, 4097, 8191, 8192, 8193, 12289, 20000])
@pytest.mark.parametrize("crowd", [1, 64])
def test_one_full_tile(n, crowd, prec, src):
    """n particles in the first of three tiles, in one cell or in all."""
    r = np.random.default_rng(n)
    cfg = _cfg((12, 4, 4))
    p = _fill(n + 7, r)
    side = 0.5 if crowd == 1 else 2.0
    for k in "xyz":
        p[k] = r.uniform(0.001, side - 0.001, n + 7)
    p["x"][n:] = r.uniform(2.1, 5.9, 7)  # the others hold a few
    _check(cfg, p, prec, src)


@pytest.mark.parametrize("prec,src", PAIRS)
@pytest.mark.parametrize("cells,n", [
    ((5, 4, 4), 0), ((5, 4, 4), 1), ((13, 9, 6), 5000),   # few tiles: places of 1024 particles
    ((64, 40, 40), 9000),      # 1600 tiles: places by wave
    ((60, 52, 44), 9000),      # 2145 tiles: counts in global memory
    ((16, 16, 16), 530001),    # places of 4096 particles
    ((80, 76, 72), 600000),    # 6840 tiles: more than the LDS counters
])
def test_many_tiles(cells, n, prec, src):
    r = np.random.default_rng(n + 1)
    cfg = _cfg(cells)
    p = _fill(n, r)
    for k, L in zip("xyz", (cfg.Lx, cfg.Ly, cfg.Lz)):
        p[k] = r.uniform(0.0, 0.999 * L, n)
    _check(cfg, p, prec, src)


@pytest.mark.parametrize("n", [100, 8192 * 2, 8192 * 2 + 1])
def test_storage_order_without_ids(n):
    r = np.random.default_rng(3)
    cfg = _cfg((8, 4, 4))
    p = _fill(n, r)
    for k, L in zip("xyz", (cfg.Lx, cfg.Ly, cfg.Lz)):
        p[k] = r.uniform(0.0, 0.999 * L, n)
    _check(cfg, p, "f64", "f64", ids=False)
