"""Species of a tile side by side or in turn (GPU) on both sides of the line
between the two (on 256 compute units): 64 and 65 tiles of few particles, 160 tiles of
899 and 901 per species, and 512 and 540 of many; as test_gpu_engine_split checks them (boxes of at
most 26 a side: 2^-23 * 26 / 0.5 = 6e-6 of a cell between FP32 positions).
"""
from __future__ import annotations

import pytest

import sputnipic_amd as S
from test_gpu_engine_split import test_split_matches_one_species as _check

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield


@pytest.mark.parametrize("push", [True, False])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("cells,counts", [
    ((32, 32, 4), (300, 0, 90)), ((20, 52, 4), (300, 90)),
    ((40, 32, 8), (160 * 899, 160 * 899)), ((40, 32, 8), (160 * 901, 160 * 901)),
    ((32, 32, 32), (512 * 2000, 512 * 6200)), ((36, 40, 24), (540 * 2000, 540 * 6200)),
])
def test_line(cells, counts, prec, push):
    _check(cells, counts, prec, push)
