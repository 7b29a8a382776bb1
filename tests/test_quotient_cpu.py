"""The residual-corrected quotients of chem_device.h against division.

Compiles a small host program over chem_device.h and compares, bit for bit:
quotient_fma with every reciprocal within one unit in the last place of 1 / b
(the device's Newton steps leave no more) against a / b, for random operands,
quotients at the edge of a binade and quotients next to the middle of two
numbers; the same for the constants the kernels divide by; and a y rounded to
binary32 against the binary32 quotient of binary32 operands."""
import subprocess

import pytest

SRC = r"""
#include <cstdio>
#include <cstring>
#include <cmath>
#include <random>
#include "chem_device.h"
using namespace lbm::chem;
static long bad = 0, seen = 0;
static void one(double a, double b)
{
    const double y0 = 1.0 / b;
    for (double y : {y0, nextafter(y0, INFINITY), nextafter(y0, -INFINITY)}) {
        ++seen;
        if (quotient_fma(a, Divisor{b, y}) != a / b) ++bad;
    }
}
static void onef(float a, float b)
{
    ++seen;
    if ((float)((double)a * (1.0 / (double)b)) != a / b) ++bad;
}
int main()
{
    std::mt19937_64 g(20261204);
    auto mant = [&] { return 1.0 + (double)(g() >> 12) * 0x1p-52; };
    auto ex = [&] { return ldexp(1.0, (int)(g() % 200) - 100); };
    auto sg = [&] { return g() & 1 ? 1.0 : -1.0; };
    for (int i = 0; i < 400000; ++i) {
        const double a = sg() * mant() * ex(), b = mant() * ex();
        one(a, b);
        const double m = mant();
        one(m * b, b);                          // quotients next to a number
        one(nextafter(m * b, 0.0), b);
        one((m + 0x1p-53 * (2.0 * (g() & 1) - 1.0)) * b, b);
        one(b * nextafter(2.0, 0.0), b);        // the top and bottom of a binade
        one(b * nextafter(1.0, 2.0), b);
        one(a, nextafter(2.0, 0.0));
        one(a, nextafter(1.0, 2.0));
        one(0.0, b);
        for (int k = 0; k < NS; ++k) one(a, W[k]);
        one(a, 3.0);
        one(a, 5.0);
        const float fa = (float)(sg() * mant() * ldexp(1.0, (int)(g() % 60) - 30)), fb = (float)(mant() * ldexp(1.0, (int)(g() % 60) - 30));
        onef(fa, fb);
        onef(fa * fb, fb);
        onef(nextafterf(fa * fb, 0.f), fb);
    }
    // the derived rows hold a2 / 3 as the run-time division gives it
    for (int k = 0; k < NS; ++k) {
        volatile double lo = NASA_LO[k][2], hi = NASA_HI[k][2], three = 3.0;
        ++seen;
        if (ROWS_LO.v[k][7] != lo / three || ROWS_HI.v[k][7] != hi / three) ++bad;
    }
    printf("%ld of %ld differ\n", bad, seen);
    return bad != 0;
}
"""


@pytest.mark.parametrize("mechdef", ["", "-DLBM_MECH_CH4_2S"])
def test_quotients_are_the_divisions(tmp_path, mechdef):
    import os
    repo = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    pkg = os.path.join(repo, "lattice-boltzmann-method_amd")
    src, exe = tmp_path / "q.cpp", tmp_path / "q"
    src.write_text(SRC)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cmd = ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas", "-D__HIP_PLATFORM_AMD__",
           f"-I{rocm}/include", f"-I{pkg}/csrc", f"-I{repo}/include"] + ([mechdef] if mechdef else [])
    subprocess.run(cmd + ["-o", str(exe), str(src), "-lm"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
