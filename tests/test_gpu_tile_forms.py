"""The column tiles, the batched solves and the placements of the m = 0
temperature solve at sizes that launch them (small groups in inverse mode take
whole mode updates instead), and the whole mode updates of more than 256
workgroups, which read the m = 0 factor from memory.

What an ensemble launches is asserted from fdns_ens_step_timed's counts.  The
tiles face the oracle directly (relative Frobenius error <= 1e-10, that of the
parity suite); forms among each other must agree bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel
from test_gpu_batch import make, states_equal

pytestmark = pytest.mark.gpu

FIELDS = ("tFR", "omgFR", "urFR", "upFR", "psi")
SCHEMES = (("CNAB2", False), ("SBDF3", True), ("ARS443", False), ("BPR353", False))


def group(Nr, Nm, n, k=0):
    """n runs of one structure (scheme k of SCHEMES)."""
    s, restart = SCHEMES[k]
    return [dict(Nr=Nr, Nm=Nm, Ra=1e5 * (1 + j % 3), Pr=(0.7, 1.0, 7.0)[j % 3], dt=1e-6, scheme=s, seed=300 + j, restart=restart)
            for j in range(n)]


@pytest.fixture
def whole_groups(fd, request):
    """Groups kept whole (a stored choice may split a large group over lanes,
    and its halves may be small)."""
    Nr = request.getfixturevalue("Nr")
    Nm = request.getfixturevalue("Nm")
    prev = fd.get_tuning(Nr, Nm)
    fd.set_tuning(Nr, Nm, **dict(prev, lane_split=0))
    yield
    fd.set_tuning(Nr, Nm, **prev)


def close(e, runs):
    e.close()
    for r in runs:
        r.close()


def launches(e):
    """Whether the next step of an ensemble of one family launches tiles (it steps)."""
    _, k = e.step_timed(1)
    pre = k["imex_pre"][1] + k["rk_pre"][1]
    mid = k["imex_mid"][1] + k["rk_mid"][1]
    assert mid > 0
    return pre > 0


# ---- the tiles against the oracle
@pytest.mark.parametrize("Nr, Nm, n", [(33, 64, 16), (97, 64, 8), (129, 64, 8)])
@pytest.mark.parametrize("k", range(4))
def test_tiles_against_oracle(fd, orc, whole_groups, Nr, Nm, n, k):
    ms = group(Nr, Nm, n, k)
    runs = [make(fd, m) for m in ms]
    e = fd.Ensemble(runs)
    e.step(3)
    got = [runs[j].get_state() for j in (0, n - 1)]
    assert launches(e)
    close(e, runs)
    for m, a in zip((ms[0], ms[-1]), got):
        o = orc.Run(Nr, Nm, m["Ra"], m["Pr"], m["dt"], m["scheme"], restart=m["restart"])
        o.set_state(*orc.seed_state(Nr, Nm, 0.35, m["seed"]))
        o.step(3)
        b = o.get_state()
        errs = {f: rel(a[f], b[f]) for f in FIELDS}
        assert max(errs.values()) <= 1e-10, errs


# ---- launch choices
DEFAULT = dict(nl_tpb=256, tile_waves=8, tile_stage=0, solve_chunk=0, tile_pf=0, lane_split=0)
STAGED = dict(nl_tpb=128, tile_waves=4, tile_stage=1, solve_chunk=8, tile_pf=1, lane_split=0)


def stepped(fd, ms, tuning, change=None, graph=True):
    Nr, Nm = ms[0]["Nr"], ms[0]["Nm"]
    prev = fd.get_tuning(Nr, Nm)
    fd.set_tuning(Nr, Nm, **tuning)
    runs = [make(fd, m) for m in ms]
    e = fd.Ensemble(runs)
    try:
        e.step(3, graph=graph)
        if change:
            fd.set_tuning(Nr, Nm, **change)
        e.step(3, graph=graph)
        out = [r.get_state() for r in runs]
        assert launches(e)
        return out
    finally:
        close(e, runs)
        fd.set_tuning(Nr, Nm, **prev)


@pytest.mark.parametrize("k", range(4))
def test_choice_change_reaches_captured_tiles(fd, k):
    ms = group(97, 64, 9, k)
    ref = stepped(fd, ms, DEFAULT)
    for got in (stepped(fd, ms, DEFAULT, change=STAGED), stepped(fd, ms, STAGED, graph=False)):
        assert all(states_equal(a, b) for a, b in zip(got, ref))


def test_solo_run_of_tiles_follows_choice(fd):
    """135 rows: past the whole mode updates also alone."""
    prev = fd.get_tuning(135, 16)
    out = []
    for change in (None, STAGED):
        fd.set_tuning(135, 16, **DEFAULT)
        r = fd.Run(135, 16, 1e5, 0.7, 1e-6, "ARS443", solver="inverse")
        r.seed(4)
        r.step(3)
        if change:
            fd.set_tuning(135, 16, **change)
        r.step(3)
        out.append(r.get_state())
        e = fd.Ensemble([r])
        assert launches(e)
        close(e, [r])
    fd.set_tuning(135, 16, **prev)
    assert states_equal(*out)


# ---- the m = 0 temperature solve: its own kernel (timed steps), the first blocks
# of the temperature-solve launch (one and two slots), the side stream
@pytest.mark.parametrize("Nr, Nm, n", [(33, 64, 16), (65, 64, 8), (97, 64, 8), (129, 64, 8), (135, 32, 2)])
@pytest.mark.parametrize("k", [0, 2])
def test_m0_placements(fd, whole_groups, Nr, Nm, n, k):
    def run(how):
        runs = []
        for m in group(Nr, Nm, n, k):
            r = fd.Run(Nr, Nm, m["Ra"], m["Pr"], m["dt"], m["scheme"], solver="inverse")
            r.seed(m["seed"])
            runs.append(r)
        e = fd.Ensemble(runs)
        if how == "timed":
            _, c = e.step_timed(6)
            assert c["solve_T"][1] > 0
        else:
            e.step(6, graph=how == "graph")
        out = [r.get_state() for r in runs]
        assert launches(e)
        close(e, runs)
        return out
    ref = run("timed")
    for how in ("eager", "graph"):
        assert all(states_equal(a, b) for a, b in zip(run(how), ref)), how


# ---- whole mode updates of 257 to 512 workgroups against the tiles
@pytest.mark.parametrize("Nr, Nm", [(17, 9), (33, 16), (48, 15), (64, 11)])
@pytest.mark.parametrize("k", [0, 3])
def test_many_workgroups(fd, whole_groups, Nr, Nm, k):
    per = 1 + (Nm + 1) // 2
    out = []
    for n, tiles in ((300 // per, False), (512 // per + 1, True)):
        assert (256 < n * per <= 512) != tiles
        runs = [make(fd, m) for m in group(Nr, Nm, n, k)]
        e = fd.Ensemble(runs)
        e.step(3)
        out.append([runs[j].get_state() for j in (0, 1, 300 // per - 1)])
        assert launches(e) == tiles
        close(e, runs)
    for a, b in zip(*out):
        assert states_equal(a, b)


# one run of many modes: 257 workgroups
@pytest.mark.parametrize("Nr", [65, 97, 128, 129, 130])
@pytest.mark.parametrize("k", [0, 2])
def test_one_run_of_many_modes(fd, Nr, k):
    out = []
    for n, tiles in ((1, False), (2, True)):
        runs = []
        for m in group(Nr, 512, n, k):
            r = fd.Run(Nr, 512, m["Ra"], m["Pr"], m["dt"], m["scheme"], solver="inverse")
            r.seed(m["seed"])
            runs.append(r)
        e = fd.Ensemble(runs)
        e.step(3)
        out.append(runs[0].get_state())
        assert launches(e) == tiles
        close(e, runs)
    assert states_equal(*out)


# ---- psi of the explicit RK path and of the step's assembly, which the other
# radial forms (up to 64 rows) write too
@pytest.mark.parametrize("Nr, Nm", [(16, 5), (33, 65), (63, 7), (64, 6), (65, 5)])
@pytest.mark.parametrize("mBC", ["NS", "SF"])
def test_psi_of_the_explicit_path(fd, orc, Nr, Nm, mBC):
    g = fd.Run(Nr, Nm, 1e5, 0.7, 1e-8, "RK4", mBC=mBC, lagpts=3)
    o = orc.Run(Nr, Nm, 1e5, 0.7, 1e-8, "RK4", mBC=mBC, lagpts=3)
    s = orc.seed_state(Nr, Nm, 0.35, 11)
    g.set_state(*s)
    o.set_state(*s)
    g.step(3)
    o.step(3)
    a, b = g.get_state()["psi"], o.get_state()["psi"]
    g.close()
    assert np.abs(b).max() > 0 and rel(a, b) <= 1e-10
