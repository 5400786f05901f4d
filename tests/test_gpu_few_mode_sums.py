"""The kinetic energies and the power budget where their kernels form the sums
over the modes themselves (at most 16 modes over the levels of a lane) and just
past it, against the oracle, from a flow with every mode at work.

Tolerance: that of the sums by a wavefront per level (test_gpu_mode_sums.py),
1e-12 for the energies of a given state, 1e-10 for the budget after a step.
"""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_mode_sums import test_mode_sums as check_sums

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nr, Nm", [(17, 8), (33, 15), (33, 16), (64, 15), (65, 7), (65, 8), (100, 7)])
@pytest.mark.parametrize("mBC", ["NS", "SF"])
def test_few_mode_sums(fd, orc, Nr, Nm, mBC):
    check_sums(fd, orc, Nr, Nm, mBC)


def test_record_is_the_diag(fd):
    """The series' row and fdns_diag give the same bits on both sides of the line."""
    for Nr, Nm in ((33, 15), (33, 16), (65, 7), (65, 8)):
        r = fd.Run(Nr, Nm, 1e5, 0.7, 1e-6, "CNAB2", n_KE=1)
        r.seed(3)
        r.step(2)
        d, row = r.diag(), r.series()[-1]
        assert np.array_equal(row, [d["t"], d["KE"], d["Nu_t"], d["Nu_b"]])
        r.close()
