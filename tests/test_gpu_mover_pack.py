"""The caller-order mover with packed fields (GPU), taken from 262144 particles
and two per node on: the same species pushed whole and in parts too small for
it end in the same bits, in both arithmetic modes, alone and fused with the
deposit (whose moments are sums in another order: 1e-12 of each array's
maximum).  Particles on the domain's edges take the clamped cells."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_bitwise, assert_close

pytestmark = pytest.mark.gpu

LIMIT = 1 << 18


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    yield
    S.set_strict_fp(False)


def _setup(cells, n, prec):
    r = np.random.default_rng(n)
    dt = np.float64 if prec == "f64" else np.float32
    L = [0.5 * c for c in cells]
    grd = S.Grid(*cells, *L, prec)
    field = S.EMField(grd, {k: r.normal(0, 0.05, grd.nn).astype(dt) for k in O.FIELD_NAMES})
    p = {k: r.uniform(0, 1, n) * l for k, l in zip("xyz", L)}
    for k, l in zip("xyz", L):
        p[k][:50], p[k][50:100] = 0.0, l
    for k in "uvw":
        p[k] = r.normal(0, 0.05, n)
    p["q"] = r.uniform(0.5, 1.5, n)
    return grd, field, {k: v.astype(dt) for k, v in p.items()}


@pytest.mark.parametrize("strict", [False, True])
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("cells,n", [((9, 7, 5), LIMIT), ((9, 7, 5), LIMIT + 77),
                                     ((60, 46, 41), LIMIT + 1), ((60, 46, 40), LIMIT + 1)])
def test_whole_equals_parts(cells, n, prec, fused, strict):
    S.set_strict_fp(strict)
    grd, field, p = _setup(cells, n, prec)
    param = S.Parameters(dt=0.25, c=1.0, NiterMover=3)

    def run(arrays, ids):
        part = S.Particles(arrays, -64.0, prec)
        if fused:
            S.mover_interp(part, field, ids, grd, param)
        else:
            S.mover_PC(part, field, grd, param)
        return part.download()

    one, two = S.InterpDensSpecies(grd), S.InterpDensSpecies(grd)
    whole = run(p, one)
    half = n // 2
    parts = [run({k: v[:half] for k, v in p.items()}, two),
             run({k: v[half:] for k, v in p.items()}, two)]
    for k in "xyzuvwq":
        assert_bitwise(whole[k], np.concatenate([q[k] for q in parts]), k)
    if fused:
        a, b = one.download(), two.download()
        for k in O.MOMENT_NAMES:
            assert_close(a[k], b[k], 1e-12, k)
