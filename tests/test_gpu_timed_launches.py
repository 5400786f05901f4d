"""What fdns_ens_step_timed times is what the steps launch, and the autotuner
chooses only among launches that a step makes.
"""
from __future__ import annotations

import pytest

from test_gpu_batch import make

pytestmark = pytest.mark.gpu

TILES = {"CNAB2": ("imex_pre", "imex_mid", "imex_post"), "ARS443": ("rk_pre", "rk_mid", "rk_post")}


def ensemble(fd, n, scheme, Nr=65, Nm=128, **kw):
    runs = [make(fd, dict(Nr=Nr, Nm=Nm, Ra=1e5 * (1 + k), Pr=0.7, dt=1e-6, scheme=scheme, seed=k + 1, **kw)) for k in range(n)]
    return runs, fd.Ensemble(runs)


# 129 modes: up to three runs take whole mode updates, more the column tiles
@pytest.mark.parametrize("n", [1, 3, 4])
@pytest.mark.parametrize("scheme", ["CNAB2", "ARS443"])
def test_classes(fd, n, scheme):
    runs, e = ensemble(fd, n, scheme)
    e.step(2)
    _, k = e.step_timed(3)
    e.close()
    for r in runs:
        r.close()
    per = 3 * (1 if scheme == "CNAB2" else 4)   # mode updates in three steps
    pre, mid, post = TILES[scheme]
    whole = n <= 3
    assert k[mid][1] == per and k[mid][0] > 0
    for c in (pre, post, "solve_T", "solve_F"):
        assert k[c][1] == (0 if whole else per), c


def test_autotune_of_whole_mode_updates(fd):
    Nr, Nm = 65, 128
    prev = fd.get_tuning(Nr, Nm)
    odd = dict(nl_tpb=256, tile_waves=[4, 8, 4, 8, 4, 8], tile_stage=[1, 0, 0, 1, 1, 0], tile_pf=[0, 1, 1, 0, 0, 1],
               solve_chunk=24, lane_split=0)
    fd.set_tuning(Nr, Nm, **odd)
    a, ea = ensemble(fd, 2, "CNAB2")
    b, eb = ensemble(fd, 2, "ARS443")
    ea.step(2)
    eb.step(2)
    for e in (ea, eb):
        chosen, report = e.autotune(steps=2)
        for k in ("tile_waves", "tile_stage", "tile_pf", "solve_chunk"):
            assert chosen[k] == odd[k], k
        assert all(v > 0 for v in report.values())
        e.close()
    fd.set_tuning(Nr, Nm, **prev)
    for r in a + b:
        r.close()
