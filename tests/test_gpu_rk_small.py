"""The explicit RK path and the schemes that are not stiffly accurate on either
side of 64 rows (up to there their radial work is one workgroup per mode),
against the oracle.

Tolerance: relative Frobenius error <= 1e-10, that of the whole parity suite
(both sides round the same sums in another order; the wall derivatives amplify
1e-15 by up to Nr^4 / 1e2).
"""
from __future__ import annotations

import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

TOL = 1e-10
FIELDS = ("tFR", "omgFR", "urFR", "upFR")


# rows around the 32-row blocks and the wavefront, groups of four rows with
# every remainder; more modes than lanes in the mean flow's sums
@pytest.mark.parametrize("Nr, Nm", [(16, 5), (17, 2), (31, 9), (32, 16), (33, 65), (50, 12), (63, 7), (64, 6), (65, 5)])
@pytest.mark.parametrize("scheme, mBC", [("RK4", "NS"), ("RK4", "SF"), ("BHR553", "NS"), ("KC343", "SF")])
def test_rows(fd, orc, Nr, Nm, scheme, mBC):
    dt = 1e-8 if scheme == "RK4" else 1e-6
    g = fd.Run(Nr, Nm, 1e5, 0.7, dt, scheme, mBC=mBC, lagpts=3)
    o = orc.Run(Nr, Nm, 1e5, 0.7, dt, scheme, mBC=mBC, lagpts=3)
    s = orc.seed_state(Nr, Nm, 0.35, 11)
    g.set_state(*s)
    o.set_state(*s)
    g.step(3)
    o.step(3)
    a, b = g.get_state(), o.get_state()
    g.close()
    errs = {k: rel(a[k], b[k]) for k in FIELDS}
    print(scheme, mBC, Nr, Nm, {k: f"{v:.1e}" for k, v in errs.items()}, flush=True)
    assert max(errs.values()) <= TOL, errs
