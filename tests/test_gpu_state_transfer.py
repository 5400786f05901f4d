"""States in and out, around the size up to which they pass through the pinned
block (a megabyte: 13107 points with the streamfunction, 16384 without), from
one thread and from several at once: the same bytes come back.
"""
from __future__ import annotations

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("tFR", "omgFR", "urFR", "upFR")


def round_trip(fd, Nr, Nm, seed):
    r = fd.Run(Nr, Nm, 1e5, 1.0, 1e-6, "CNAB2")
    rng = np.random.default_rng(seed)
    s = [np.asfortranarray(rng.standard_normal((Nm + 1, Nr)) + 1j * rng.standard_normal((Nm + 1, Nr))) for _ in FIELDS]
    r.set_state(*s)
    a = r.get_state()
    r.close()
    return all(np.array_equal(a[f], x) for f, x in zip(FIELDS, s)) and not a["psi"].any()


@pytest.mark.parametrize("Nr, Nm", [(16, 1), (64, 203), (66, 199), (65, 204), (64, 255), (65, 255)])
def test_round_trip(fd, Nr, Nm):
    assert round_trip(fd, Nr, Nm, 1)


def test_round_trip_threads(fd):
    ok = []
    def work(k):
        ok.extend(round_trip(fd, 33, 16 + k, 10 * k + j) for j in range(8))
    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert len(ok) == 32 and all(ok)
