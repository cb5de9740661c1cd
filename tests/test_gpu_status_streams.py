"""Reports of particles that left the grid, with work in flight on another stream
(GPU): synchronous calls on one stream report their own particles, whatever an
asynchronous call on another sets meanwhile or later, in the same thread and in
threads that come after it; the check of that other stream reports it once.
"""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S
from sputnipic_amd._capi import check, lib

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield
    S.set_async(False)
    check(lib().spic_synchronize(), "wait")
    try:
        S.check_domain()
    except S.SpicError:
        pass


class _Setup:
    def __init__(self):
        self.grd = S.Grid(8, 4, 4, 4.0, 2.0, 2.0, "f64")
        self.field = S.EMField(self.grd, {k: np.zeros(self.grd.nn) for k in O.FIELD_NAMES})
        self.param = S.Parameters(dt=0.25, c=1.0)
        self.good, self.bad = self._part(100, 0.01), self._part(100, 100.0)
        self.long = self._part(400000, 0.01, niter=40000)

    @staticmethod
    def _part(n, u, niter=3):
        p = {k: np.full(n, 1.0) for k in "xyz"}
        p.update({k: np.full(n, u) for k in "uvw"})
        p["q"] = np.ones(n)
        return S.Particles(p, 1.0, "f64", NiterMover=niter)

    def move(self, part, stream=None):
        g, f, s, p = (self.grd.c_struct(), self.field.c_struct(), part.c_struct(),
                      self.param.push())
        check(lib().spic_mover_pc(C.byref(g), C.byref(f), C.byref(s), C.byref(p),
                                  stream.ptr if stream else None), "mover_PC")

    def late(self, stream):
        """Asynchronously on `stream`: some hundred milliseconds of work, then
        particles that leave the grid."""
        S.set_async(True)
        for _ in range(3):
            self.move(self.long, stream)
        self.move(self.bad, stream)
        S.set_async(False)


def _check(stream):
    check(lib().spic_check_domain(stream.ptr), "check")


@pytest.mark.parametrize("wait", ["check", "stream", "none"])
def test_calls_beside_another_streams(wait):
    st, a, b = _Setup(), S.Stream(), S.Stream()
    st.move(st.good, b)
    st.late(a)
    st.move(st.good, b)       # while the other stream works
    if wait == "check":
        with pytest.raises(S.SpicError):
            _check(a)
        _check(a)
    elif wait == "stream":
        a.synchronize()
    else:                     # known to have ended, but not to this library
        ev = S.Event()
        ev.record(a)
        end = S.Event()
        end.record(a)
        ev.elapsed_ms(end)
    for _ in range(3):
        st.move(st.good, b)
    with pytest.raises(S.SpicError):
        st.move(st.bad, b)
    st.move(st.good, a)
    st.move(st.good, b)
    a.synchronize()


def test_threads_that_follow():
    st, a, b = _Setup(), S.Stream(), S.Stream()
    seen = []

    def first():
        st.late(a)
        try:
            st.move(st.good, b)
        except S.SpicError as e:
            seen.append(e)

    def then():
        try:
            for _ in range(3):
                st.move(st.good, b)
            a.synchronize()
            for _ in range(3):
                st.move(st.good, b)
        except S.SpicError as e:
            seen.append(e)

    for work in (first, then):
        t = threading.Thread(target=work)
        t.start()
        t.join()
    assert not seen


def test_check_clears_before_other_streams():
    st, streams = _Setup(), [S.Stream() for _ in range(6)]
    for a in streams:
        with pytest.raises(S.SpicError):
            st.move(st.bad, a)
        with pytest.raises(S.SpicError):
            _check(a)
        for b in streams:
            st.move(st.good, b)
    S.set_async(True)
    for a in streams:  # more streams than are followed one by one
        st.move(st.bad, a)
    S.set_async(False)
    check(lib().spic_synchronize(), "wait")
    for b in streams:
        st.move(st.good, b)
