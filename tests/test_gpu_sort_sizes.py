"""particle_sort at sizes around its workgroups (GPU), both precisions, which
gather two and four arrays at a time: every array bit for bit in the oracle's
order, the allocation-free entry point included."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_bitwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1025, 70001])
def test_sort_sizes(n, prec, noalloc):
    S.set_async(False)
    cfg = O.GemConfig(nxc=9, nyc=6, nzc=5, Lx=4.5, Ly=3.0, Lz=2.5, npcelx=[1] * 4,
                      npcely=[1] * 4, npcelz=[1] * 4)
    r = np.random.default_rng(n)
    dt = np.float64 if prec == "f64" else np.float32
    p = {k: (r.uniform(0, 1, n) * L).astype(dt)
         for k, L in zip("xyz", (cfg.Lx, cfg.Ly, cfg.Lz))}
    p.update({k: r.normal(0, 1, n).astype(dt) for k in "uvwq"})
    st = O.State(cfg, prec, build_ic=False)
    st.parts = [{k: v.copy() for k, v in p.items()}]
    st.particle_sort(0, 2)
    grd = S.Grid(cfg.nxc, cfg.nyc, cfg.nzc, cfg.Lx, cfg.Ly, cfg.Lz, prec)
    part = S.Particles(p, 1.0, prec)
    g, s = grd.c_struct(), part.c_struct()
    call = S._capi.lib().spic_particle_sort_noalloc if noalloc else (
        S._capi.lib().spic_particle_sort)
    assert call(C.byref(g), 2, C.byref(s), None) == 0
    got = part.download()
    for k in "xyzuvwq":
        assert_bitwise(got[k], st.parts[0][k], k)
