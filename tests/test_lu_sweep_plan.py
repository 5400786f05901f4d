"""The barriers of the LU-mode solves: every wavefront of a workgroup passes as
many, for every matrix order, also in a launch with more wavefronts than the
matrix has rows for (the m = 0 system beside the coupled ones).

The plan is plain C++ (csrc/fdns_sweep.h); a small program goes over it as the
kernel's loops do.
"""
from __future__ import annotations

import os
import subprocess

from conftest import REPO

PROGRAM = r"""
#include <cstdio>
#include "fdns_sweep.h"
using namespace fdns;
// the barriers of one sweep: two per pair taken part in, then one each up to the last
static int barriers(LuxShare s)
{
    int b = 0;
    for (int k = 0; k < s.mine; ++k) b += 2;
    for (int k = 2 * s.mine; k < 2 * s.pairs; ++k) ++b;
    return b;
}
int main()
{
    int bad = 0;
    for (int n = 4; n <= 1026; ++n)
        for (int wide = 0; wide < 2; ++wide) {
            const int nblk = lux_blocks(n), waves = lux_waves(wide ? 2 * n : n);
            for (int wv = 0; wv < waves; ++wv) {
                const LuxShare d = lux_backward(nblk, wv);
                bool ok = d.mine >= 0 && d.mine <= d.pairs && barriers(d) == 2 * d.pairs &&
                          // every block at or above the wavefront's rows is one it takes part in
                          2 * d.mine >= nblk - LUX_WB * wv;
                for (int b0 = 0; b0 <= nblk; ++b0) {
                    const LuxShare u = lux_forward(nblk, b0, wv);
                    const int top = LUX_WB * (wv + 1) < nblk ? LUX_WB * (wv + 1) : nblk;
                    ok = ok && u.mine >= 0 && u.mine <= u.pairs && barriers(u) == 2 * u.pairs && 2 * u.mine >= top - b0;
                }
                if (!ok && bad++ < 5) std::printf("n %d, %d wavefronts, wavefront %d\n", n, waves, wv);
            }
        }
    std::printf("%d\n", bad);
    return bad != 0;
}
"""


def test_every_wavefront_passes_the_same_barriers(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(REPO, "falcon-dns_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
