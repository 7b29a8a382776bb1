"""The kernels' quotients on the device against division, bit for bit.

quotient_check.hip runs divisor() and quot() of chem_device.h, so the hardware's
own reciprocal is in it.  Operands: random ones, quotients one part in 2^106 off
the middle of two numbers, powers of two, and the constants the kernels divide
by.  Where the device's 1 / b is the correctly rounded one the quotient must be
a / b; it may be another only for divisors just below a power of two (their 1 / b
lies within 2^-88 of a middle), and the quotient is then a neighbour of a / b."""
import ctypes
import os

import numpy as np
import pytest

from lbm_amd import capi

pytestmark = pytest.mark.gpu

U54 = np.uint64((1 << 54) - 1)


def near_middles(n, rng):
    """Odd 53-bit B and A with A / B next to an odd 54-bit number over 2^k."""
    B = (rng.integers(1 << 52, 1 << 53, n, dtype=np.uint64)) | np.uint64(1)
    B[:2000] = np.uint64((1 << 53) - 1) - np.uint64(2) * np.arange(2000, dtype=np.uint64)
    B[2000:4000] = np.uint64((1 << 52) + 1) + np.uint64(2) * np.arange(2000, dtype=np.uint64)
    inv = np.ones_like(B)
    for _ in range(7):  # B^-1 modulo 2^64
        inv *= np.uint64(2) - B * inv
    a, b = [], []
    for sign in (1, -1):
        M = (inv if sign > 0 else np.uint64(0) - inv) & U54  # M B = sign modulo 2^54
        keep = M >= np.uint64(1 << 53)
        for m, d in zip(M[keep][:40000].tolist(), B[keep][:40000].tolist()):
            num = (m * d - sign) >> 54
            assert (m * d - sign) & ((1 << 54) - 1) == 0
            if num < 1 << 53:
                a.append(float(num))
                b.append(float(d))
    return np.array(a), np.array(b)


def test_device_quotients_are_the_divisions():
    lib = ctypes.CDLL(os.path.join(os.path.dirname(capi.library_path()), "libquotient_check.so"))
    rng = np.random.default_rng(20261205)
    a0, b0 = near_middles(200000, rng)
    b1 = rng.uniform(1, 2, 400000) * 2.0 ** rng.integers(-100, 100, 400000)
    a1 = rng.choice([-1, 1], b1.size) * rng.uniform(1, 2, b1.size) * 2.0 ** rng.integers(-100, 100, b1.size)
    ones = 2.0 - 2.0 ** -52 * np.arange(1, 5001)
    a2 = np.concatenate([2.0 ** rng.integers(-30, 30, ones.size), rng.uniform(1, 2, ones.size)])
    const = np.concatenate([np.tile([3.0, 5.0, 12000.0], 1), rng.uniform(1, 60, 997)])
    a = np.concatenate([a0, a1, a2, np.repeat(rng.uniform(-1, 1, 100), const.size)])
    b = np.concatenate([b0, b1, ones, ones, np.tile(const, 100)])
    q, y = np.empty_like(a), np.empty_like(a)
    dp = [x.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for x in (a, b, q, y)]
    assert lib.quotient_check(*dp, ctypes.c_int64(a.size)) == 0
    rounded = y == 1.0 / b
    assert np.array_equal(q[rounded], (a / b)[rounded])
    mant = np.frexp(b[~rounded])[0]  # in [1/2, 1)
    print(f"{(~rounded).sum()} of {b.size} reciprocals are the other neighbour", flush=True)
    assert np.all(mant >= 1.0 - 1024 * 2.0 ** -53)
    other = ~rounded & (q != a / b)
    assert np.all(np.abs(q - a / b)[other] <= np.spacing(np.abs(a / b)[other]))
