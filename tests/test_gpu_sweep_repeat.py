"""The solves by sweeps that are done again with masks and divisions, because
their solution leaves the range in which a reciprocal stands for the division.

A fresh IMEX step of a flow at rest is linear in the state, and a power of two
scales every operation of it exactly: a state scaled out of that range must
give the scaled fields, bit for bit.  The mean temperature (its walls, at 1 and
0, are far below an ulp of both states) takes the one-wavefront sweeps in their
forms -- one run, one to three 64-row slots; a few runs, the factor read from
memory; many runs, the column tiles with the sweep in the temperature-solve
launch (up to 100 rows) or k_m0; LU mode -- and in LU mode the other modes take
the coupled solves.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = ([(Nr, 16, 1, "inverse") for Nr in (16, 33, 64, 65, 97, 129, 130)] + [(64, 16, 40, "inverse")] +
         [(33, 64, 16, "inverse"), (65, 64, 8, "inverse"), (97, 64, 8, "inverse"), (129, 64, 8, "inverse")] +
         [(Nr, 16, 1, "lu") for Nr in (16, 33, 65, 129, 193)])


def step(fd, Nr, Nm, n, solver, mean, scale):
    x = np.cos(np.pi * (Nr - 1 - np.arange(Nr)) / (Nr - 1))
    rng = np.random.default_rng(Nr)
    runs = []
    for k in range(n):
        r = fd.Run(Nr, Nm, 1e5, 0.7, 1e-6, "CNAB2", solver=solver)
        s = [np.zeros((Nm + 1, Nr), dtype=complex, order="F") for _ in range(4)]
        for f in (0, 1):
            c = rng.standard_normal((Nm + 1, 3)) + 1j * rng.standard_normal((Nm + 1, 3))
            p = (c @ np.stack([1 + 0 * x, x, x * x])) * (1 - x * x)
            s[f][...] = (p if not mean else 0.0)
        s[0][0], s[1][0] = (scale * (2.0 + x) if mean else 0.0), 0.0
        s[0][1:] *= scale
        s[1][1:] *= scale
        r.set_state(*s)
        runs.append(r)
    e = fd.Ensemble(runs)
    try:
        e.step(1)
        return [r.get_state() for r in runs]
    finally:
        e.close()
        for r in runs:
            r.close()


@pytest.mark.parametrize("Nr, Nm, n, solver", FORMS)
def test_mean_temperature(fd, Nr, Nm, n, solver):
    a, b = step(fd, Nr, Nm, n, solver, True, 2.0**500), step(fd, Nr, Nm, n, solver, True, 2.0**950)
    for x, y in zip(a, b):
        assert np.isfinite(y["tFR"]).all() and np.abs(y["tFR"][0]).max() > 2.0**900
        assert np.array_equal(x["tFR"] * 2.0**450, y["tFR"])


@pytest.mark.parametrize("Nr", [16, 33, 64, 65, 129, 193])
def test_coupled_solves(fd, Nr):
    a, b = step(fd, Nr, 16, 1, "lu", False, 1.0), step(fd, Nr, 16, 1, "lu", False, 2.0**-850)
    for k in ("tFR", "omgFR", "urFR", "upFR", "psi"):
        x, y = a[0][k][1:], b[0][k][1:]
        assert x.any() and np.array_equal(x * 2.0**-850, y), k
