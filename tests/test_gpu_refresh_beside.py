"""An asynchronous refresh of the chemistry network must go on beside large steps.

The steps' kernels fill the registers and LDS of every CU.  Training kernels whose
blocks need a whole CU start only between two step kernels: 100 iterations then
took some 15 times as long beside 256x128x128 steps as by themselves.  Blocks that
fit into the place of a step kernel's block share the CUs; sharing them evenly
with the step's two streams is a factor of three, and twice that is the bar.
"""
import time

import pytest

from lbm_amd import cases
from lbm_amd.capi import LBM_FP32_SHIFTED, LBM_MODE_FUSED, MixtureLattice

pytestmark = pytest.mark.gpu


def test_refresh_goes_on_beside_large_steps():
    n = (256, 128, 128)
    lat = MixtureLattice(*n, *cases.UNITS_FLAME, reaction=True, precision=LBM_FP32_SHIFTED, mode=LBM_MODE_FUSED)
    lat.load_case(cases.mixing_layer(*n, T_fuel=300.0, T_ox=1200.0, U_s=0.02))
    lat.Init()
    lat.calculate_moment()
    cells = n[0] * n[1] * n[2]
    lat.surrogate_capture(cells, 8)
    lat.step(4)
    lat.surrogate_capture_stop()
    lat.surrogate_train(400, batch=4096, lr=1e-3, seed=1)
    lat.surrogate_enable(True, audit_stride=64, audit_tol=0.5)
    lat.surrogate_capture(2 * cells, 1 << 30)
    lat.step(2)
    lat.surrogate_refresh(100, batch=4096, lr=3e-4, seed=2)
    t0 = time.perf_counter()
    lat.surrogate_refresh(100, batch=4096, lr=3e-4, seed=3)
    alone = time.perf_counter() - t0
    beside = []
    for seed in (4, 5):
        lat.sync()
        t0 = time.perf_counter()
        lat.surrogate_refresh_async(100, batch=4096, lr=3e-4, seed=seed)
        for _ in range(60):
            lat.step(1)
            lat.sync()
            if lat.surrogate_refresh_poll(wait=False):
                break
        else:
            lat.surrogate_refresh_poll(wait=True)
        beside.append(time.perf_counter() - t0)
    lat.close()
    assert min(beside) < 6 * alone, (beside, alone)
