"""A load of more tiles than a small workgroup counts (6840, counted and placed
by workgroups of 1024 threads from 4194304 particles on; one particle fewer by
waves): the particles come back to the last bit, and the engine's deposit of
them equals the caller-order deposit (1e-12 of each array's maximum in FP64,
1e-5 in FP32, whose engine holds fixed-point positions)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_close

pytestmark = pytest.mark.gpu

LINE = 256 * 1024 * 16


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [LINE - 1, LINE, LINE + 5])
def test_many_tiles_of_many_particles(n, prec):
    S.set_async(False)
    S.set_strict_fp(False)
    r = np.random.default_rng(n)
    cells = (80, 76, 72)
    L = [0.5 * c for c in cells]
    dt = np.float64 if prec == "f64" else np.float32
    p = {k: (r.random(n) * 0.999 * l).astype(dt) for k, l in zip("xyz", L)}
    for k in "uvw":
        p[k] = (r.random(n) - 0.4).astype(dt)
    p["q"] = (r.random(n) + 0.5).astype(dt)
    grd = S.Grid(*cells, *L, prec)
    part, got, want = S.Particles(p, 1.0, prec), S.InterpDensSpecies(grd), S.InterpDensSpecies(grd)
    S.interpP2G(part, want, grd)
    eng = S.Engine(grd, 1, set_moments=True)
    try:
        eng.load(0, part)
        eng.deposit([got])
        eng.store(0, part)
    finally:
        eng.close()
    back = part.download()
    for k in "xyzuvwq":
        if prec == "f32" and k in "xyz":
            assert np.all(np.abs(back[k].astype(np.float64) - p[k]) <= 1e-5), k
        else:
            assert np.array_equal(back[k], p[k]), k
    a, b = got.download(), want.download()
    for k in O.MOMENT_NAMES:
        assert_close(a[k], b[k], 1e-12 if prec == "f64" else 1e-5, k)
