"""The field operators at the edges of their kernels' tiles (4 x 4 x 16
cells): grids around one and two tiles per axis, bit for bit against the
oracle for every periodicity, the ghosts written by the same pass; and
results in the memory of an input, which the operators take."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_bitwise
from test_gpu_field import PERIODICITIES, _device, _state

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 3), (3, 4, 15), (4, 3, 16), (5, 9, 17), (8, 7, 33)]


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("per", PERIODICITIES)
def test_hat_and_image(per, shape):
    st = _state(per, shape)
    grd, field, ids, sp, _ = _device(st)
    net = S.InterpDensNet(grd)
    S.sumOverSpecies(net, ids, grd, st.cfg.ns)
    S.interpN2Crho_net(net, grd, sp)
    rhon, rhoc = st.rhoc_from_rhon(st.sum_species()["rhon"])
    assert_bitwise(net.d["rhon"].download(), rhon, "rhon")
    assert_bitwise(net.rhoc.download(), rhoc, "rhoc")
    aux = S.InterpDensAux(grd)
    S.calculateHatDensities(aux, net, ids, field, grd, sp)
    want, got = st.hat_densities(rhoc), aux.download()
    for n in ("rhoh", "Jxh", "Jyh", "Jzh"):
        assert_bitwise(got[n], want[n], n)
    g = st.grid
    m = 3 * (g.nxn - 2) * (g.nyn - 2) * (g.nzn - 2)
    vec = np.random.default_rng(5).normal(0, 1e-2, m)
    dv, im = S.DeviceArray.from_numpy(vec), S.DeviceArray(m, np.float64)
    S.MaxwellImage(im, dv, field, ids, grd, sp)
    want = st.maxwell_image(vec)
    assert_bitwise(im.download(), want, "image")
    S.MaxwellImage(dv, dv, field, ids, grd, sp)
    assert_bitwise(dv.download(), want, "image in place")


def test_hat_current_in_a_tensors_memory():
    st = _state((1, 0, 1), (9, 6, 18))
    grd, field, ids, sp, _ = _device(st)
    net, aux = S.InterpDensNet(grd), S.InterpDensAux(grd)
    _, rhoc = st.rhoc_from_rhon(st.sum_species()["rhon"])
    net.rhoc.upload(rhoc)
    aux.J["Jyh"] = ids[1].d["pxy"]
    S.calculateHatDensities(aux, net, ids, field, grd, sp)
    want, got = st.hat_densities(rhoc), aux.download()
    for n in ("rhoh", "Jxh", "Jyh", "Jzh"):
        assert_bitwise(got[n], want[n], n)
