"""fdns_diag only reads a run: a thread that asks an ensemble's members for
their energies while another steps the ensemble leaves every state as it was.

The members are past the whole-mode updates (more than 256 workgroups of two
modes), so their steps pass right-hand sides and solutions through the run's
work arrays, which the sums of the diagnostics must not touch.
"""
from __future__ import annotations

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("tFR", "omgFR", "urFR", "upFR", "psi")
CALLS, MOST = 30, 400   # questions to ask, calls of 50 steps at most


def stepped(fd, scheme, steps):
    """States and energies after `steps` calls of 50 steps; steps None: as many
    as it takes another thread to ask CALLS questions meanwhile."""
    runs, stop, calls = [], threading.Event(), [0]
    for k in range(6):
        r = fd.Run(65, 128, 1e5 * (1 + k), 0.7, 1e-6, scheme, solver="inverse")
        r.seed(k + 1)
        runs.append(r)
    e = fd.Ensemble(runs)

    def ask():
        while not stop.is_set():
            runs[calls[0] % 6].diag()
            calls[0] += 1

    t = threading.Thread(target=ask)
    try:
        e.step(2)
        if steps is None:
            t.start()
            steps = 0
            while steps < MOST and calls[0] < CALLS:
                e.step(50)
                steps += 1
            stop.set()
            t.join()
            assert calls[0] >= CALLS
        else:
            for _ in range(steps):
                e.step(50)
        return steps, [r.get_state() for r in runs], [r.diag() for r in runs]
    finally:
        stop.set()
        if t.is_alive():
            t.join()
        e.close()
        for r in runs:
            r.close()


@pytest.mark.parametrize("scheme", ["CNAB2", "ARS443"])
def test_diag_during_steps(fd, scheme):
    steps, a, da = stepped(fd, scheme, None)
    _, b, db = stepped(fd, scheme, steps)
    for x, y in zip(a, b):
        for k in FIELDS:
            assert np.array_equal(x[k], y[k]), k
    assert da == db
