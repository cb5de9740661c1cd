"""How exactly FP32 engines sum their moments (GPU): many particles of one cell,
of a tile that the grid's end leaves one cell wide, and of every cell alike,
against the FP64 oracle's deposit of the very particles that the engine holds.

Here a sum in FP32 runs over at most 128 terms (half of 64 batches at four per
cell; of a clump at most 24 per batch) before it goes on in FP64, and the tile's sum
is rounded to FP32 once.  With rounding errors of 0.41 * 2^-24 (rms) of the running
value that is 0.41 sqrt(128 / 3) / sqrt(2) + 0.41 = 2.3 * 2^-24 of the sum of the
terms' magnitudes; a term's own ten roundings average out over the many terms of a
node.  Bound: 8 * 2^-24 of the largest sum of magnitudes.  One FP32 chain over
all 32768 particles of a cell is off by 0.41 sqrt(32768 / 3) = 43 * 2^-24.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S

pytestmark = pytest.mark.gpu

TOL = 8 * 2.0 ** -24


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield
    S.set_strict_fp(False)


def _oracle(cfg, p):
    st = O.State(cfg, "f64", build_ic=False)
    st.parts = [p]
    st.zero_moments(0)
    st.interp_p2g(0)
    return st.moments[0]


@pytest.mark.parametrize("push", [False, True])
@pytest.mark.parametrize("opts", [
    dict(), dict(strict=True), dict(positions=S.SPIC_POS_FLOAT), dict(particles_per_thread=2),
    dict(tile=(8, 4, 4))])
@pytest.mark.parametrize("cells,box,n", [
    ((12, 4, 4), (0, 0, 0, 1, 1, 1), 32768),   # one cell of a full tile
    ((5, 5, 5), (4, 4, 4, 1, 1, 1), 32768),    # the one cell of the last tile
    ((5, 4, 4), (4, 0, 0, 1, 4, 4), 8192),     # a tile one cell thick
    ((8, 4, 4), (0, 0, 0, 8, 4, 4), 128 * 256),
])
def test_fp32_sums(cells, box, n, opts, push):
    opts = dict(opts)
    S.set_strict_fp(opts.pop("strict", False))
    d = 0.5
    cfg = O.GemConfig(nxc=cells[0], nyc=cells[1], nzc=cells[2], Lx=d * cells[0],
                      Ly=d * cells[1], Lz=d * cells[2], npcelx=[1] * 4, npcely=[1] * 4,
                      npcelz=[1] * 4)
    r = np.random.default_rng(11)
    p = {}
    for a, k in enumerate("xyz"):  # well inside their cells: the push leaves them there
        c = r.integers(box[a], box[a] + box[3 + a], n)
        p[k] = (c + r.uniform(0.2, 0.8, n)) * d
    for k in "uvw":
        p[k] = r.normal(0.05, 0.1, n)
    p["q"] = r.uniform(0.5, 1.5, n) / n
    p = {k: v.astype(np.float32) for k, v in p.items()}
    grd = S.Grid(*cells, cfg.Lx, cfg.Ly, cfg.Lz, "f32")
    part, mom = S.Particles(p, 1.0, "f32"), [S.InterpDensSpecies(grd)]
    back = S.Particles({k: np.zeros(n) for k in p}, 1.0, "f64")  # positions to the last bit
    eng = S.Engine(grd, 1, set_moments=True, **opts)
    try:
        eng.load(0, part)
        if push:
            eng.phase(S.EMField(grd), mom, S.Parameters(dt=0.05, c=1.0, NiterMover=3))
        else:
            eng.deposit(mom)
        eng.store(0, back)
    finally:
        eng.close()
    held, got = back.download(), mom[0].download()
    want = _oracle(cfg, held)
    size = _oracle(cfg, {k: np.abs(v) for k, v in held.items()})
    for k in O.MOMENT_NAMES:
        off = np.max(np.abs(np.asarray(got[k]) - want[k])) / np.max(size[k])
        assert off <= TOL, (k, off / 2.0 ** -24)
