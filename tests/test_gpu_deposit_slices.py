"""Caller-order deposits of species of more than 2^24 particles, which go through
tiles in slices (GPU), against the oracle as in test_gpu_deposit_limits.  Up to
2^31 - 1 particles the slices are checked when the library is compiled.
"""
from __future__ import annotations

import pytest

import sputnipic_amd as S
from test_gpu_deposit_limits import _big

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("n", [(1 << 24) - 1, 1 << 24, (1 << 24) + 1, (1 << 24) + 70001])
def test_slices(n, fused):
    _big((9, 6, 5), n, "uniform", "f32", fused)
