"""lbm_step's three streams (chemistry, mixture energy, species) against the
serial calls, through the C ABI.

Every kernel has to see the inputs that the five calls issued one by one give
it, so the bar is bitwise equality of all fluid cells after each step.  The
cases are those where an order could go wrong: each execution mode and
precision, with and without chemistry, an inflow and an outflow whose sweeps
follow the energy stream, two charges on a grid of a few wavefronts, and a
binary32 grid large enough for the energy part to have a stream of its own there.
"""
import time

import numpy as np
import pytest

from lbm_amd import cases
from lbm_amd.capi import (LBM_FP32_SHIFTED, LBM_FP64, LBM_MODE_FUSED, LBM_MODE_INPLACE, LBM_MODE_STRICT, POP_F, POP_G,
                          LbmError)
from mode_compare import assert_same, make, snapshot

pytestmark = pytest.mark.gpu

BUILD = {
    "flame": lambda: cases.premixed_flame_1d(70, 3, 4),
    "layer": lambda: cases.mixing_layer(6, 12, 5, T_fuel=300.0, T_ox=1200.0, U_s=0.02, delta=3.0),
    "box": lambda: cases.reacting_box(16, 12, 10, T_K=1300.0, amp_T=0.1, amp_u=0.01),
    "large": lambda: cases.reacting_box(53, 52, 51, T_K=1300.0, amp_T=0.1, amp_u=0.01),  # 157 thousand cells
}


@pytest.mark.parametrize("reaction", [False, True])
@pytest.mark.parametrize("case,mode,precision", [
    ("flame", LBM_MODE_STRICT, LBM_FP64), ("flame", LBM_MODE_FUSED, LBM_FP64),
    ("layer", LBM_MODE_STRICT, LBM_FP32_SHIFTED), ("layer", LBM_MODE_FUSED, LBM_FP32_SHIFTED),
    ("layer", LBM_MODE_INPLACE, LBM_FP32_SHIFTED), ("box", LBM_MODE_FUSED, LBM_FP64),
    ("box", LBM_MODE_INPLACE, LBM_FP64), ("large", LBM_MODE_FUSED, LBM_FP32_SHIFTED),
    ("large", LBM_MODE_INPLACE, LBM_FP32_SHIFTED), ("large", LBM_MODE_STRICT, LBM_FP32_SHIFTED)])
def test_overlapped_step_matches_serial_calls(case, mode, precision, reaction):
    fl = BUILD[case]()
    F = fl["type"].ravel() == 0
    ov, ser = make(fl, mode, precision, reaction), make(fl, mode, precision, reaction)
    try:
        print(f"{case} mode {mode} precision {precision} reaction {reaction}", flush=True)
        for step in range(1, 5):
            ov.step(1)
            ser.Collide_Species()
            ser.Collide()
            ser.Streaming()
            ser.TMS_BC()
            ser.calculate_moment()
            assert_same(snapshot(ov, F), snapshot(ser, F), f"step {step}")
        ov.step(3)
        ser.step(3)
        assert_same(snapshot(ov, F), snapshot(ser, F), "three steps in one call")
    finally:
        ov.close()
        ser.close()


def test_refused_step_leaves_the_energy_populations(monkeypatch):
    """An in-place step whose species collide is refused (LBM_AMD_LOW_MAX below
    one species' floor pairs) must leave the populations as the refused serial
    call does: the energy populations stream only in a step that goes through."""
    monkeypatch.setenv("LBM_AMD_LOW_MAX", "100")
    fl = cases.reacting_box(6, 5, 4, T_K=1300.0, amp_T=0.1, amp_u=0.01, X={"O2": 0.3, "N2": 0.7})
    ov, ser = (make(fl, LBM_MODE_INPLACE, LBM_FP64, False) for _ in range(2))
    try:
        before = ov.get_populations(POP_G)
        with pytest.raises(LbmError, match="SPECIES_MIN"):
            ov.step(1)
        with pytest.raises(LbmError, match="SPECIES_MIN"):
            ser.Collide_Species()
        assert (ser.get_populations(POP_G) == before).all()
        assert (ov.get_populations(POP_G) == before).all()
        assert (ov.get_populations(POP_F) == ser.get_populations(POP_F)).all()
    finally:
        ov.close()
        ser.close()


@pytest.mark.parametrize("reaction", [False, True])
@pytest.mark.parametrize("mode", [LBM_MODE_FUSED, LBM_MODE_STRICT, LBM_MODE_INPLACE])
def test_small_steps_pay_for_no_stream(mode, reaction, monkeypatch):
    """A step of a small binary32 grid takes no longer than the serial calls': the
    two are the same kernels, so anything over a sixth is the streams' events (they
    cost half as much again when every step used all three streams)."""
    fl = cases.reacting_box(6, 17, 9, T_K=1300.0, amp_T=0.05, amp_u=0.01)
    lats = []
    try:
        for env in ("1", "0"):
            monkeypatch.setenv("LBM_AMD_OVERLAP", env)
            lats.append(make(fl, mode, LBM_FP32_SHIFTED, reaction))
        times = [[], []]
        for _ in range(15):
            for lat, t in zip(lats, times):
                lat.step(5)
                lat.sync()
                t0 = time.perf_counter()
                lat.step(20)
                lat.sync()
                t.append(time.perf_counter() - t0)
        ov, serial = (float(np.median(t)) for t in times)
        assert ov < serial * 7 / 6, (ov / 20, serial / 20)
    finally:
        for lat in lats:
            lat.close()
