"""Re-sorts of tiles at the edges of what a workgroup stages (GPU): ranks per
cell around the slot tables (256 in FP32, 512 in FP64; half that for 8x4x4
tiles), particles per tile around the staged chunk and the largest staged
tile.  A sort moves values: they come back to the last bit (fixed-point
positions within 1e-5), and the deposit after it matches the oracle's (1e-13 in
FP64; 5e-5 in FP32, where positions are rounded to float)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("tile", [(4, 4, 4), (8, 4, 4)])
@pytest.mark.parametrize("crowd,n", [(1, 127), (1, 128), (1, 129), (1, 255), (1, 256), (1, 257),
                                     (1, 511), (1, 512), (1, 513), (64, 4095), (64, 4096),
                                     (64, 4097), (64, 12288), (64, 12289), (64, 17000)])
def test_sort_of_a_full_tile(crowd, n, tile, prec):
    S.set_async(False)
    S.set_strict_fp(False)
    r = np.random.default_rng(n)
    cfg = O.GemConfig(nxc=16, nyc=4, nzc=4, Lx=8.0, Ly=2.0, Lz=2.0, npcelx=[1] * 4,
                      npcely=[1] * 4, npcelz=[1] * 4)
    dt = np.float64 if prec == "f64" else np.float32
    side = 0.5 if crowd == 1 else 2.0
    p = {k: r.uniform(0.001, side - 0.001, n + 9) for k in "xyz"}
    p["x"][n:] = r.uniform(2.1, 7.9, 9)
    p.update({k: r.normal(0, 0.1, n + 9) for k in "uvw"})
    p["q"] = r.uniform(0.5, 1.5, n + 9)
    p = {k: v.astype(dt) for k, v in p.items()}
    grd = S.Grid(cfg.nxc, cfg.nyc, cfg.nzc, cfg.Lx, cfg.Ly, cfg.Lz, prec)
    part, mom = S.Particles(p, 1.0, prec), [S.InterpDensSpecies(grd)]
    eng = S.Engine(grd, 1, tile=tile, set_moments=True)
    try:
        eng.load(0, part)
        for _ in range(2):
            eng.sort()
        eng.deposit(mom)
        eng.store(0, part)
    finally:
        eng.close()
    got, mom = part.download(), mom[0].download()
    for k in "xyzuvwq":
        if k in "xyz" and prec == "f32":
            assert np.all(np.abs(got[k].astype(np.float64) - p[k]) <= 1e-5), k
        else:
            assert np.array_equal(got[k], p[k]), k
    st = O.State(cfg, prec, build_ic=False)
    st.parts = [got]
    st.zero_moments(0)
    st.interp_p2g(0)
    for k in O.MOMENT_NAMES:
        assert_close(mom[k], st.moments[0][k], 1e-13 if prec == "f64" else 5e-5, k)
