"""The deposit of small species (GPU): counts around the 32 particles of a
wave, cells that change with every particle or never, faces and ghost cells,
and both sides of the line to the deposit through tiles (16384 particles, eight
per tile); and the fused push, which then runs as two kernels.

Moments within 1e-13 of each array's maximum of the oracle's in FP64 (the same
terms in another order) and 1e-5 of the FP32 oracle, which sums in float;
particle state bit for bit in strict arithmetic.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from helpers import assert_bitwise, assert_close
from test_gpu_deposit_tiles import _pair

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield
    S.set_strict_fp(False)


def _moments(st, ids, prec):
    got = ids.download()
    for k in O.MOMENT_NAMES:
        assert_close(got[k], st.moments[0][k], 1e-13 if prec == "f64" else 1e-5, k)


@pytest.mark.parametrize("strict", [True, False])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["uniform", "sorted", "one_cell", "faces"])
@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 63, 64, 65, 1000])
def test_small_deposit(n, kind, prec, strict):
    _, st, grd, _, part, ids, _ = _pair(n, kind, prec)
    S.set_strict_fp(strict)
    S.interpP2G(part, ids, grd)
    st.zero_moments(0)
    st.interp_p2g(0)
    _moments(st, ids, prec)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,kind", [(16383, "uniform"), (16384, "uniform"), (16384, "sorted"),
                                    (33 * 512, "one_cell"), (33 * 512 + 1, "one_cell")])
def test_both_sides_of_the_line(n, kind, prec):
    _, st, grd, _, part, ids, _ = _pair(n, kind, prec)
    S.interpP2G(part, ids, grd)
    st.zero_moments(0)
    st.interp_p2g(0)
    _moments(st, ids, prec)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [1, 33, 700])
def test_small_fused(n, prec):
    _, st, grd, field, part, ids, param = _pair(n, "uniform", prec)
    S.set_strict_fp(True)
    S.mover_interp(part, field, ids, grd, param)
    st.zero_moments(0)
    st.mover_pc(0)
    st.interp_p2g(0)
    got = part.download()
    for k in "xyzuvw":
        assert_bitwise(got[k], st.parts[0][k], k)
    _moments(st, ids, prec)
