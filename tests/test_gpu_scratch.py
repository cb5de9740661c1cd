"""Scratch memory of the caller-order calls (GPU): kept in a bounded pool between
calls, given back on request, taken beside a capture on another stream, and not
needed while captured: the results stay the same."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
import sputnipic_amd as S
from helpers import assert_close
from sputnipic_amd._capi import check, lib

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield
    S.set_async(False)
    S.release_scratch()


def _state(n, cells=(40, 40, 40)):
    grd = S.Grid(*cells, *(0.5 * c for c in cells), "f64")
    r = np.random.default_rng(n)
    p = {k: r.uniform(0.1, 0.5 * c - 0.1, n) for k, c in zip("xyz", cells)}
    p.update({k: r.normal(0, 0.01, n) for k in "uvw"})
    p["q"] = r.uniform(0.5, 1.5, n)
    field = S.EMField(grd, {k: r.normal(0, 0.01, grd.nn) for k in O.FIELD_NAMES})
    return grd, field, S.Particles(p, 1.0, "f64"), S.InterpDensSpecies(grd), S.Parameters(dt=0.01)


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_given_back():
    grd, field, part, ids, param = _state(8_000_000)
    S.mover_interp(part, field, ids, grd, param)  # loads the kernels
    S.release_scratch()
    before = _free()
    S.mover_interp(part, field, ids, grd, param)
    kept = before - _free()
    assert 8 * 8_000_000 <= kept <= 512 * MIB
    S.release_scratch()
    assert before - _free() <= 2 * MIB
    S.mover_interp(part, field, ids, grd, param)  # and taken again
    assert before - _free() <= 512 * MIB
    S.release_scratch()
    S.release_scratch()  # nothing left


@pytest.mark.parametrize("n", [20000, 300000])
def test_beside_a_capture(n):
    """An asynchronous call on one stream while another stream is captured."""
    grd, field, part, ids, param = _state(n)
    _, _, twin, ids2, _ = _state(n)
    S.release_scratch()
    g, f, p, k = grd.c_struct(), field.c_struct(), part.c_struct(), param.push()
    m, m2, p2 = ids.c_struct(), ids2.c_struct(), twin.c_struct()
    a, b = S.Stream(), S.Stream()
    graph = S.Graph(a)
    with graph:
        check(lib().spic_zero_moments(C.byref(g), C.byref(m), a.ptr), "zero")
        check(lib().spic_mover_interp(C.byref(g), C.byref(f), C.byref(p), C.byref(m),
                                      C.byref(k), a.ptr), "captured")
        check(lib().spic_zero_moments(C.byref(g), C.byref(m2), b.ptr), "zero")
        check(lib().spic_mover_interp(C.byref(g), C.byref(f), C.byref(p2), C.byref(m2),
                                      C.byref(k), b.ptr), "beside")
    b.synchronize()
    for _ in range(3):
        graph.launch()
        a.synchronize()
        one, two = part.download(), twin.download()
        for c in "xyzuvw":
            assert np.array_equal(one[c], two[c]), c
        got, want = ids.download(), ids2.download()
        for c in O.MOMENT_NAMES:
            assert_close(got[c], want[c], 1e-12, c)
        S.set_async(False)
        ids2.upload({c: np.zeros(grd.nn) for c in O.MOMENT_NAMES})
        S.mover_interp(twin, field, ids2, grd, param)
        S.set_async(True)
    S.set_async(False)
    S.check_domain()
    graph.close()
