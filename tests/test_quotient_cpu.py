"""The residual-corrected quotients of chem_device.h against division, bit for bit.

Host builds of the device's arithmetic.  With the correctly rounded reciprocal
quotient_fma has to be a / b for random operands, for quotients at the edges of a
binade and for quotients as close to the middle of two numbers as they come: B odd
with 53 bits and M = -+B^-1 modulo 2^54, A = (M B +- 1) / 2^54, so that A / B is
M / 2^54 give or take one part in 2^106.  With the reciprocal's other neighbour
some of those must differ (or the operands are not what they are meant to be).
divisor() has to give the correctly rounded reciprocal from a hardware one that is
up to 2^-22 off, but for divisors just below a power of two; there the quotient
may be a neighbour of a / b, as a power of two over 2 - 2^-52 is.  Also the
constants the kernels divide by, and the binary32 quotients through a binary64
reciprocal."""
import pytest

from device_arithmetic import run

BODY = r"""
static long bad = 0, seen = 0, near_mid = 0, other_side = 0, off = 0;
static void expect(bool ok)
{
    ++seen;
    if (!ok) ++bad;
}
static void one(double a, double b)
{
    expect(quotient_fma(a, Divisor{b, 1.0 / b}) == a / b);
    const Divisor d = divisor(b);
    const double q = quot(a, d);
    if (d.y == 1.0 / b) {
        expect(q == a / b);
    } else {  // less than 2^-42 below a power of two, and q a neighbour at most
        int e;
        ++off;
        expect(std::fabs(std::frexp(b, &e)) >= 1.0 - 0x1p-42);
        expect(q == a / b || q == nextafter(a / b, INFINITY) || q == nextafter(a / b, -INFINITY));
    }
}
static void onef(float a, float b)
{
    expect((float)((double)a * (1.0 / (double)b)) == a / b);
}
int main()
{
    std::mt19937_64 g(20261204);
    auto mant = [&] { return 1.0 + (double)(g() >> 12) * 0x1p-52; };
    auto ex = [&] { return ldexp(1.0, (int)(g() % 200) - 100); };
    auto sg = [&] { return g() & 1 ? 1.0 : -1.0; };
    for (int i = 0; i < 400000; ++i) {
        rcp_error = ldexp(1.0, -22 - (int)(g() % 8));
        const double a = sg() * mant() * ex(), b = mant() * ex();
        one(a, b);
        const double m = mant();
        one(m * b, b);                          // quotients next to a number
        one(nextafter(m * b, 0.0), b);
        one(b * nextafter(2.0, 0.0), b);        // the top and bottom of a binade
        one(b * nextafter(1.0, 2.0), b);
        one(a, nextafter(2.0, 0.0));
        one(a, nextafter(1.0, 2.0));
        one(0.0, b);
        for (int k = 0; k < NS; ++k) one(a, W[k]);
        one(a, 3.0);
        one(a, 5.0);
        // next to a middle: the first thousands of divisors at both ends of a binade
        uint64_t B = (g() >> 12) | (1ull << 52) | 1;
        if (i < 4000) B = (1ull << 53) - 1 - 2 * i;
        else if (i < 8000) B = (1ull << 52) + 1 + 2 * (i - 4000);
        uint64_t inv = 1;
        for (int k = 0; k < 7; ++k) inv *= 2 - B * inv;  // B^-1 modulo 2^64
        for (int s = -1; s <= 1; s += 2) {
            const uint64_t M = (s > 0 ? inv : -inv) & ((1ull << 54) - 1);
            if (M < (1ull << 53)) continue;
            const unsigned __int128 p = (unsigned __int128)M * B - s;
            expect((uint64_t)(p & ((1ull << 54) - 1)) == 0);
            const uint64_t A = (uint64_t)(p >> 54);
            if (A >= (1ull << 53)) continue;
            ++near_mid;
            one((double)A, (double)B);
            for (double to : {0.0, (double)INFINITY})
                other_side += quotient_fma((double)A, Divisor{(double)B, nextafter(1.0 / (double)B, to)}) !=
                              (double)A / (double)B;
        }
        const float fa = (float)(sg() * mant() * ldexp(1.0, (int)(g() % 60) - 30)), fb = (float)(mant() * ldexp(1.0, (int)(g() % 60) - 30));
        onef(fa, fb);
        onef(fa * fb, fb);
        onef(nextafterf(fa * fb, 0.f), fb);
    }
    // the divisors just below a power of two, over powers of two
    for (int k = 1; k < 4000; ++k) one(1.0, 2.0 - 0x1p-52 * k);
    // the derived rows hold a2 / 3 as the run-time division gives it
    for (int k = 0; k < NS; ++k) {
        volatile double lo = NASA_LO[k][2], hi = NASA_HI[k][2], three = 3.0;
        expect(ROWS_LO.v[k][7] == lo / three && ROWS_HI.v[k][7] == hi / three);
    }
    printf("%ld of %ld differ; %ld next to a middle, %ld of them wrong through a neighbour; %ld reciprocals off\n", bad, seen,
           near_mid, other_side, off);
    return bad != 0 || near_mid < 100000 || other_side < near_mid / 10 || off == 0;
}
"""


@pytest.mark.parametrize("mechdef", ["", "-DLBM_MECH_CH4_2S"])
def test_quotients_are_the_divisions(tmp_path, mechdef):
    run(tmp_path, BODY, [mechdef] if mechdef else [])
