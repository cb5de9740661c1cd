"""Status words of threads that come and go (GPU): every thread's synchronous
calls report their own particles, also on words that an earlier thread gave
back."""
from __future__ import annotations

import threading

import pytest

import sputnipic_amd as S
from test_gpu_status import _setup

pytestmark = pytest.mark.gpu


def test_words_given_back_start_clean():
    S.set_async(False)
    good, bad = _setup()
    log = []

    def work(calls):
        for c in calls:
            try:
                (bad if c else good)()
                log.append((c, 0))
            except S.SpicError:
                log.append((c, 1))

    for calls in ((0,), (1,), (0, 1, 0), (0,), (1, 0), (0, 0)) * 4:
        t = threading.Thread(target=work, args=(calls,))
        t.start()
        t.join()
    many = [threading.Thread(target=work, args=((0, 1, 0),)) for _ in range(8)]
    for t in many:
        t.start()
    for t in many:
        t.join()
    assert len(log) == 4 * 10 + 8 * 3
    assert all(c == e for c, e in log)
