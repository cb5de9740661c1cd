"""What a call reports about particles that left the grid (GPU): a synchronous
call reports its own, whatever earlier calls left; an asynchronous one leaves
it for the check, which reports once; each thread, and a graph's replays, have
theirs."""
from __future__ import annotations

import threading

import numpy as np
import pytest

import oracle as O
import sputnipic_amd as S

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _modes():
    S.set_async(False)
    S.set_strict_fp(False)
    yield
    S.set_async(False)
    try:
        S.check_domain()
    except S.SpicError:
        pass


def _setup():
    grd = S.Grid(8, 4, 4, 4.0, 2.0, 2.0, "f64")
    z = np.zeros(grd.nn)
    field = S.EMField(grd, {k: z for k in O.FIELD_NAMES})
    param = S.Parameters(dt=0.25, c=1.0)

    def part(u):
        n = 100
        p = {k: np.full(n, 1.0) for k in "xyz"}
        p.update({k: np.full(n, u) for k in "uvw"})
        p["q"] = np.ones(n)
        return S.Particles(p, 1.0, "f64")

    good, bad = (lambda: S.mover_PC(part(0.01), field, grd, param)), (
        lambda: S.mover_PC(part(100.0), field, grd, param))
    return good, bad


def test_synchronous_calls_report_their_own():
    good, bad = _setup()
    for _ in range(2):
        good()
        with pytest.raises(S.SpicError):
            bad()
        good()
    with pytest.raises(S.SpicError):
        bad()
    with pytest.raises(S.SpicError):
        S.check_domain()  # still there
    S.check_domain()
    good()


def test_asynchronous_calls_leave_it_for_the_check():
    good, bad = _setup()
    S.set_async(True)
    bad()
    good()
    with pytest.raises(S.SpicError):
        S.check_domain()
    S.check_domain()
    bad()
    S.set_async(False)
    good()  # a synchronous call starts anew
    S.check_domain()


def test_threads_have_their_own():
    good, bad = _setup()
    seen = []

    def work():
        try:
            bad()
        except S.SpicError:
            seen.append(1)

    t = threading.Thread(target=work)
    t.start()
    t.join()
    assert seen == [1]
    S.check_domain()
    good()


def test_replays_do_not_reach_later_calls():
    grd = S.Grid(8, 4, 4, 4.0, 2.0, 2.0, "f64")
    good, bad = _setup()
    n = 100
    p = {k: np.full(n, 1.0) for k in "xyzuvw"}
    p["u"] = np.full(n, 0.01)
    p["v"] = p["w"] = np.zeros(n)
    p["q"] = np.ones(n)
    part, ids = S.Particles(p, 1.0, "f64"), [S.InterpDensSpecies(grd)]
    field = S.EMField(grd, {k: np.zeros(grd.nn) for k in O.FIELD_NAMES})
    param = S.Parameters(dt=0.25, c=1.0)
    eng = S.Engine(grd, 1, set_moments=True)
    stream = S.Stream()
    try:
        eng.load(0, part)
        S.set_async(True)
        g = S.Graph(stream)
        with g:
            for _ in range(2):
                eng.phase(field, ids, param, stream)
        field.d["Ex"].upload(np.full(grd.nn, 1e6))  # the replay throws them out
        g.launch()
        stream.synchronize()
        S.set_async(False)
        good()
        with pytest.raises(S.SpicError):
            bad()
        good()
        g.close()
    finally:
        S.set_async(False)
        eng.close()
