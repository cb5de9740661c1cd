"""MaxwellImage on both sides of the line between its kernel's narrow and wide
tiles (4 x 4 x 16 and 8 x 4 x 16 cells, wide from 256 of them on), ragged grids
included: bit for bit against the oracle, every periodicity."""
from __future__ import annotations

import numpy as np
import pytest

import sputnipic_amd as S
from helpers import assert_bitwise
from test_gpu_field import PERIODICITIES, _device, _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(136, 60, 16), (64, 64, 32), (73, 33, 33), (129, 3, 161)])
@pytest.mark.parametrize("per", PERIODICITIES)
def test_image_of_wide_tiles(per, shape):
    S.set_async(False)
    S.set_strict_fp(False)
    st = _state(per, shape)
    grd, field, ids, sp, _ = _device(st)
    g = st.grid
    m = 3 * (g.nxn - 2) * (g.nyn - 2) * (g.nzn - 2)
    vec = np.random.default_rng(5).normal(0, 1e-2, m)
    dv, im = S.DeviceArray.from_numpy(vec), S.DeviceArray(m, np.float64)
    S.MaxwellImage(im, dv, field, ids, grd, sp)
    assert_bitwise(im.download(), st.maxwell_image(vec), "image")
