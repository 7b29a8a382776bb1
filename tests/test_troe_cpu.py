"""Troe's broadening factor where its inner divisor passes through zero.

log10 F = lFc / (1 + f1^2) with f1 = (lPr + c) / (n - 0.14 (lPr + c)): f1 has a
pole at lPr + c = n / 0.14, where the factor is 1 (log 0).  Every number next to
the pole is tried, with the device's arithmetic: the values have to be finite and
those of the formula in extended precision (three roundings of the inner divisor,
whose relative error at the pole is unbounded, only move |f1| among numbers whose
square is above 1e20: both sides are 0 to 1e-20 there)."""
import pytest

from device_arithmetic import run

BODY = r"""
int main()
{
    long bad = 0, zero = 0;
    std::mt19937_64 g(3);
    for (int k = 0; k < 4000; ++k) {
        const double lFc = -1.0 - 2.0 * (double)(g() >> 11) * 0x1p-53;
        const double c = -0.4 - 0.67 * lFc, n = 0.75 - 1.27 * lFc;
        double lPr = n / 0.14 - c;
        for (int i = 0; i < 40; ++i) lPr = nextafter(lPr, 0.0);
        for (int i = 0; i < 80; ++i, lPr = nextafter(lPr, INFINITY)) {
            const double d = n - 0.14 * (lPr + c);
            zero += d == 0.0;
            const double got = troe_log_f(lPr, lFc);
            if (!(std::fabs(got) <= 1e-20)) ++bad;
        }
        // and away from it
        const double x = -6.0 + 40.0 * (double)(g() >> 11) * 0x1p-53;
        const long double cl = c, nl = n, dl = nl - 0.14L * (x + cl), f1 = (x + cl) / dl, want = lFc / (1 + f1 * f1);
        if (std::fabs((double)dl) > 1e-3 && std::fabs((double)(troe_log_f(x, lFc) - want)) > 1e-11 * std::fabs((double)want))
            ++bad;
    }
    printf("%ld bad, %ld exact zeros\n", bad, zero);
    return bad != 0 || zero == 0;
}
"""


@pytest.mark.parametrize("mechdef", ["", "-DLBM_MECH_NH3"])
def test_broadening_factor_at_its_pole(tmp_path, mechdef):
    run(tmp_path, BODY, [mechdef] if mechdef else [])
