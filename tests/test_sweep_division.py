"""The division of the solves' backward sweeps (csrc/fdns_sweep.h): by the
reciprocal, its quotient is that of the division, bit for bit, wherever the
solve does not repeat itself -- divisor in rcp_safe's range, quotient usual --
for ordinary numbers, mantissas next to 1 and 2, subnormals, overflowing
quotients, infinities and NaN; and a solve is repeated only outside the range
that ordinary runs keep to.  (LU mode's block sweeps take div_by for the stored
value too: there a quotient at half the smallest subnormal may be zero.)
"""
from __future__ import annotations

import os
import re
import subprocess

from conftest import REPO

CSRC = os.path.join(REPO, "falcon-dns_amd", "csrc")

PROGRAM = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <limits>
#include "fdns_sweep.h"
using namespace fdns;
static uint64_t s = 88172645463325252ull;
static uint64_t next() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; }
static double bits(uint64_t b) { double x; std::memcpy(&x, &b, 8); return x; }
// a number of exponent e; every fourth mantissa next to 1 or 2
static double num(int e)
{
    uint64_t m = next() >> 12;
    if ((next() & 3) == 0) m = (next() & 1) ? (next() & 15) : (1ull << 52) - 1 - (next() & 15);
    return std::ldexp(bits((next() & (1ull << 63)) | (1023ull << 52) | m), e);
}
int main()
{
    long bad = 0, kept = 0, again = 0;
    auto check = [&](double x, double d) {
        if (!rcp_safe(d)) return;
        const double q = div_last(x, d, 1.0 / d), w = x / d;
        if (!usual(q)) { ++again; return; }
        ++kept;
        if (!(q == w) && bad++ < 5) std::printf("%a / %a: %a, not %a\n", x, d, q, w);
    };
    for (int k = 0; k < 20000000; ++k) {
        check(num((int)(next() % 121) - 60), num((int)(next() % 121) - 60));
        if (k % 4 == 0) check(num((int)(next() % 2100) - 1074), num((int)(next() % 798) - 399));
    }
    const double inf = std::numeric_limits<double>::infinity(), nan = std::nan("");
    const double odd[] = {0.0, inf, -inf, nan, 1.7e308, -1.7e308, 5e-324, -5e-324, 2.2e-308, 1e-290, 1e290};
    for (double x : odd)
        for (int k = 0; k < 2000; ++k) check(x, num((int)(next() % 798) - 399));
    // what must be repeated, and what must not
    const long n = again;
    check(inf, 2.0); check(nan, 2.0); check(1.7e308, 0.5);
    if (again != n + 3) { std::printf("an overflow passes as usual\n"); ++bad; }
    for (double x : {0.0, 1e-30, 1.0, 1e20, 1e120, 1e-120}) if (!usual(x)) { std::printf("%g is not usual\n", x); ++bad; }
    std::printf("%ld kept, %ld repeated, %ld wrong\n", kept, again, bad);
    return bad != 0;
}
"""


def test_quotients(tmp_path):
    src, exe = tmp_path / "div.cpp", tmp_path / "div"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout


def test_every_solve_by_sweeps_is_checked():
    """Each place that sweeps looks over its solution, and has the solve that
    stands in for it."""
    src = open(os.path.join(CSRC, "fdns_kernels.hip")).read()
    for name in ("void m0_solve(", "void k_m0(", "void fu_lu("):
        body = src[src.index(name):]
        body = body[:body.index("\n}\n")]
        sweeps = [m.end() for m in re.finditer(r"lu_solve_wave<|lu_wave_bwd<", body)]
        assert sweeps and body.index("lu_wave_usual<") > max(sweeps), name
        assert name == "void fu_lu(" or "lu_wave_exact(" in body, name
    assert src.count("if (odd) fu_lu_exact(") == 2   # the m = 0 temperature, and psi
    body = src[src.index("void k_solve_lu("):]
    body = body[:body.index("\n}\n")]
    assert body.index("lu_solve_reg(") < body.index("usual(x0.x)") < body.index("lu_solve_exact(")
