"""The field operators on a grid of more than a million cells along x and one
along y and z (GPU), whose image takes its tiles in several launches.  Bit for bit
against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_bitwise
from test_gpu_field import _device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per", [(1, 0, 1), (0, 1, 0)])
def test_long_grid(per):
    S.set_async(False)
    S.set_strict_fp(False)
    cfg = O.GemConfig(ns=1, nxc=1100003, nyc=1, nzc=1, Lx=1100003 * 0.5, Ly=0.5, Lz=0.5,
                      npcelx=[1] * 4, npcely=[1] * 4, npcelz=[1] * 4, PERIODICX=bool(per[0]),
                      PERIODICY=bool(per[1]), PERIODICZ=bool(per[2]))
    st = O.State(cfg, "f64", build_ic=False)
    r = np.random.default_rng(7)
    for n in O.FIELD_NAMES:
        st.fields[n][:] = r.normal(0, 1e-2, st.nn)
    for n in O.MOMENT_NAMES:
        st.moments[0][n][:] = r.normal(0, 1e-2, st.nn)
    grd, field, ids, sp, _ = _device(st)
    rhoc = r.normal(0, 1e-2, st.ncell)
    net, aux = S.InterpDensNet(grd), S.InterpDensAux(grd)
    net.rhoc.upload(rhoc)
    S.calculateHatDensities(aux, net, ids, field, grd, sp)
    want, got = st.hat_densities(rhoc), aux.download()
    for n in ("rhoh", "Jxh", "Jyh", "Jzh"):
        assert_bitwise(got[n], want[n], n)
    g = st.grid
    vec = r.normal(0, 1e-2, 3 * (g.nxn - 2) * (g.nyn - 2) * (g.nzn - 2))
    dv, im = S.DeviceArray.from_numpy(vec), S.DeviceArray(len(vec), np.float64)
    S.MaxwellImage(im, dv, field, ids, grd, sp)
    assert_bitwise(im.download(), st.maxwell_image(vec), "image")
