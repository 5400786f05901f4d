"""The solve kernels at the sizes where their tiles end, against the oracle.

Tolerance: relative Frobenius error <= 1e-10, that of the whole parity suite:
the LU-mode solves take dgetrs' operations in its order, so only the radial
transforms' rounding (~1e-15 relative, amplified by the wall derivatives)
separates the two.
"""
from __future__ import annotations

import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

TOL = 1e-10
FIELDS = ("tFR", "omgFR", "urFR", "upFR", "psi")


def check(fd, orc, Nr, Nm, scheme, steps, solver, seed=7, **kw):
    g = fd.Run(Nr, Nm, 1e5, 0.7, 1e-6, scheme, solver=solver, **kw)
    g.seed(seed)
    g.step(steps)
    a = g.get_state()
    g.close()
    o = orc.Run(Nr, Nm, 1e5, 0.7, 1e-6, scheme, **kw)
    o.set_state(*orc.seed_state(Nr, Nm, 0.35, seed))
    o.step(steps)
    b = o.get_state()
    errs = {k: rel(a[k], b[k]) for k in FIELDS}
    print(scheme, Nr, Nm, solver, {k: f"{v:.1e}" for k, v in errs.items()}, flush=True)
    assert max(errs.values()) <= TOL, errs


# matrix orders N and 2N around the column block (8 rows) and the rows of one
# wavefront (128): a last block of 1..8 rows, one wavefront exactly, one row more
@pytest.mark.parametrize("Nr", [5, 12, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 193])
@pytest.mark.parametrize("mBC", ["NS", "SF"])
def test_lu_mode_orders(fd, orc, Nr, mBC):
    check(fd, orc, Nr, 5, "CNAB2", 3, "lu", mBC=mBC)


# the boundary-row order of the IMEXRK operators (other pivot rows lead)
@pytest.mark.parametrize("Nr", [12, 64, 65, 129])
def test_lu_mode_orders_imexrk(fd, orc, Nr):
    check(fd, orc, Nr, 5, "ARS443", 2, "lu")


# matrix orders N and 2N around the factorisation's panels (16 columns), its
# rows per lane (64 each, up to 320 in one wavefront's registers) and the
# multi-wavefront panels above (one row per thread to 512, three beyond)
@pytest.mark.parametrize("Nr", [16, 17, 48, 80, 95, 160, 161, 256, 257])
def test_lu_factor_orders(fd, orc, Nr):
    check(fd, orc, Nr, 3, "CNAB2", 2, "lu")
