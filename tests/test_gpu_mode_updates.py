"""The whole mode updates against the column tiles.

A run is stepped alone (one mode per workgroup), in an ensemble of a few (two
modes per workgroup) and in one that fills the chip several times (the column
tiles, which the parity suite holds against the oracle).  Both forms take the
same operations in the same order, so the states must agree bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("tFR", "omgFR", "urFR", "upFR", "psi")


def states(fd, Nr, Nm, scheme, n, at, steps, **kw):
    """State and history of the members in at of n runs stepped together."""
    runs = []
    for k in range(n):
        r = fd.Run(Nr, Nm, 1e5 * (1.0 + k), 0.7, 1e-6 / (1 + k % 3), scheme, solver="inverse", **kw)
        r.seed(3 + k % 5)
        runs.append(r)
    if n == 1:
        runs[0].step(steps)
    else:
        e = fd.Ensemble(runs)
        e.step(steps)
        e.close()
    out = [(runs[k].get_state(), runs[k].history()) for k in at]
    for r in runs:
        r.close()
    return out


# rows around the 32-row blocks and the wavefront, the largest order, groups of
# four rows with every remainder; one mode beside m = 0, odd and even numbers
@pytest.mark.parametrize("Nr, Nm", [(5, 1), (16, 6), (17, 9), (33, 16), (48, 15), (64, 11), (65, 14), (97, 21), (128, 10),
                                    (129, 13), (130, 12)])
@pytest.mark.parametrize("scheme, buo", [("CNAB2", "IMP"), ("SBDF3", "IMP"), ("ARS443", "IMP"), ("BPR353", "EXP")])
def test_mode_updates_match_tiles(fd, Nr, Nm, scheme, buo):
    kw = dict(buo=buo, lagpts=3 if Nr < 17 else 14, restart=scheme == "SBDF3")
    few = 257 // (Nm + 1) + 1                                       # more than one mode per CU
    many = (512 if Nr <= 64 else 256) // (1 + (Nm + 1) // 2) + 1    # past the mode kernels' last launch
    assert few < many
    one = states(fd, Nr, Nm, scheme, 1, (0,), 3, **kw)
    two = states(fd, Nr, Nm, scheme, few, (0, few - 1), 3, **kw)
    tiles = states(fd, Nr, Nm, scheme, many, (0, few - 1), 3, **kw)
    assert np.isfinite(tiles[1][0]["tFR"]).all()
    for got, want in ((one[0], tiles[0]), (two[0], tiles[0]), (two[1], tiles[1])):
        for a, b, names in zip(got, want, (FIELDS, tuple(want[1]))):
            for k in names:
                assert np.array_equal(a[k], b[k]), k
