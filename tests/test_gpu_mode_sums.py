"""The sums over modes behind the kinetic energies and the power budget (one
wavefront per level) at the numbers of modes and levels where their lanes and
workgroups end, against the oracle, from a flow with every mode at work.

Tolerance: the kinetic energies of a given state are sums of positive terms
(relative error of some N Nm rounding errors: 1e-12); the budget follows a
step and takes the parity suite's 1e-10.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def flow(orc, Nr, Nm):
    """The seeded state with smooth profiles of every mode added."""
    rng = np.random.default_rng(Nr + 1000 * Nm)
    x = np.cos(np.pi * (Nr - 1 - np.arange(Nr)) / (Nr - 1))
    out = []
    for f in orc.seed_state(Nr, Nm, 0.35, 3, amp=1e-1):
        c = rng.standard_normal((Nm + 1, 4)) + 1j * rng.standard_normal((Nm + 1, 4))
        c[0].imag = 0.0
        p = (c[:, :3] @ np.stack([1 + 0 * x, x, x * x])) * (1 - x * x) / (1.0 + np.arange(Nm + 1))[:, None]
        out.append(np.asfortranarray(f + 0.1 * p))
    return out


@pytest.mark.parametrize("Nr, Nm", [(12, 2), (33, 63), (34, 64), (35, 65), (69, 128), (98, 192)])
@pytest.mark.parametrize("mBC", ["NS", "SF"])
def test_mode_sums(fd, orc, Nr, Nm, mBC):
    kw = dict(mBC=mBC, lagpts=3)
    g = fd.Run(Nr, Nm, 1e5, 0.7, 1e-7, "CNAB2", n_KE=1, **kw)
    o = orc.Run(Nr, Nm, 1e5, 0.7, 1e-7, "CNAB2", **kw)
    s = flow(orc, Nr, Nm)
    g.set_state(*s)
    o.set_state(*s)
    a, b = g.diag(), o.diag()
    for k in ("KE", "KE_r", "KE_phi"):
        assert abs(a[k] - b[k]) <= 1e-12 * abs(b[k]), k
    g.step(1)
    o.step(1)
    (bg, ug), (bo, uo) = g.budget(), o.budget()
    for k in ("KE_mean", "vis", "buo"):
        assert abs(bg[k] - bo[k]) <= 1e-10 * abs(bo[k]), k
    err = float(np.abs(ug[:, 1] - uo[:, 1]).max())   # the Reynolds stress, on the balance's scale
    assert err <= 1e-10 * float(np.abs(uo[:, 1:]).max())
    g.close()
