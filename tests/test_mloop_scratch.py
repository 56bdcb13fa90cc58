"""The LDS that the m-loop kernels ask for holds every partial sum that their
dense products store, at each n_r and thread count a launch can have
(collocation 8 .. 256, integration 8 .. 257).  The largest index is found
from the stores of the three product routines, group by group, and compared
with the layout that sizes the launch; the host compiler evaluates both, so
no GPU takes part."""
import os
import subprocess

import pytest

from helpers import ROOT

HIPCC = "/opt/rocm/bin/hipcc"

SOURCE = r"""
#include "pz_mphase.h"
struct Top { size_t n = 0; constexpr void at(size_t i) { n = i + 1 > n ? i + 1 : n; } };
// block_matvec_rc: red[a RS + (cg - 1) R RPT + ru RPT + r] for 0 < cg < CG
constexpr size_t matvec_top(int nrow, int ncol, int nt, int rpt, int nmat)
{
    Top t;
    const int R = (nrow + rpt - 1) / rpt, CG = nt / R < ncol ? nt / R : ncol, RS = (CG > 1 ? CG - 1 : 0) * R * rpt;
    for (int cg = 1; cg < CG; cg++) t.at((nmat - 1) * RS + (cg - 1) * R * rpt + (R - 1) * rpt + rpt - 1);
    return t.n;
}
// MatAhead::apply: red[a RS + cg RW + ru RPT + r] for cg < CG
constexpr size_t ahead_top(int nrow, int ncol, int nt, int rpt, int nmat)
{
    Top t;
    const int R = (nrow + rpt - 1) / rpt, CG = nt / R < ncol ? nt / R : ncol, RW = R * rpt;
    for (int cg = 0; cg < CG; cg++) t.at((nmat - 1) * CG * RW + cg * RW + (R - 1) * rpt + rpt - 1);
    return t.n;
}
// SharedMv::run: red[(a CG + cg) ldm + 4 ru + r] for cg < CG
constexpr size_t shared_top(int N, int nt, int nvec)
{
    Top t;
    const int ldm = (N + 3) & ~3, RU = ldm / 4, CG = shared_groups(N, nt);
    for (int cg = 0; cg < CG; cg++) t.at(((nvec - 1) * CG + cg) * ldm + 4 * (RU - 1) + 3);
    return t.n;
}
constexpr size_t allotted(int N, int nt, bool rad, bool integ)
{
    return (mloop_lds(N, nt, rad, integ) - MpLayout(N, rad).red) / sizeof(cd);
}
// the first n_r of [lo, hi] whose products leave the scratch; 0: none
constexpr int collocation(int lo, int hi, bool rad, bool narrow)
{
    for (int N = lo; N <= hi; N++) {
        const int nt = narrow ? 256 : mloop_threads(N);
        const size_t have = allotted(N, nt, rad, false);
        if (matvec_top(N, N, nt, 2, 2) > have || matvec_top(N, N, nt, 2, 1) > have) return N;
        if (matvec_top(2 * N, N, nt, 1, 1) > have || ahead_top(2 * N, N, nt, 1, 1) > have) return N;
        if (ahead_top(N, N, nt, 2, 1) > have) return N;
    }
    return 0;
}
constexpr int integration(int lo, int hi)
{
    for (int N = lo; N <= hi; N++) {
        const int nt = mloop_threads(N);
        const size_t have = allotted(N, nt, true, true);
        if (matvec_top(N, N, nt, 2, 1) > have || ahead_top(N, N, nt, 2, 2) > have) return N;
        if (ahead_top(N, N, nt, 1, 1) > have || shared_top(N, nt / 2, 3) > have || shared_top(N, nt, 1) > have) return N;
    }
    return 0;
}
static_assert(CHECK == 0);
"""


@pytest.mark.parametrize("check", [
    "collocation(8, 256, true, false)", "collocation(8, 256, false, false)", "collocation(66, 128, true, true)",
    "collocation(66, 128, false, true)", "integration(8, 257)"])
def test_products_stay_inside_the_scratch(check, tmp_path):
    src = tmp_path / "scratch.hip"
    src.write_text(SOURCE.replace("CHECK", check))
    r = subprocess.run([HIPCC, "-std=c++17", "-x", "hip", "--offload-host-only", "-fsyntax-only",
                        "-fconstexpr-steps=10000000", "-I" + os.path.join(ROOT, "pizza_amd", "csrc"),
                        "-I" + os.path.join(ROOT, "include"), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
