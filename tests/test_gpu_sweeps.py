"""TMS_BC's outflow and inflow sweeps at the edges of their launches against
the oracle, through the C ABI.

Both sweeps share two launches where their cells lie apart and have two each
where they are near, blocks take 16 entries (8 with many species) and 64, and
the two kinds of entry do not share a block of targets.  So the cases are
entry counts around 16 and 64, interfaces five cells apart and nearer, and both
kinds of ghost: the state after TMS_BC and after the moments that follow, the
device re-seeded from the oracle before each call (tolerance of the other
per-call comparisons).
"""
import pytest

from lbm_amd import cases
from lbm_amd.capi import POP_F, POP_G
from mode_compare import seed_gpu_from_oracle
from test_gpu_multi import TOL, check_state, fluid, pair, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nx,ny,nz", [
    ("flame", 12, 3, 5), ("flame", 12, 5, 13), ("flame", 8, 8, 8),
    ("flame", 6, 3, 4), ("flame", 4, 4, 4), ("flame", 5, 5, 13),
    ("channel", 5, 6, 3), ("channel", 9, 7, 13)])
def test_sweeps_match_oracle(kind, nx, ny, nz):
    if kind == "flame":
        fl = cases.premixed_flame_1d(nx, ny, nz)
    else:
        fl = cases.reacting_channel(nx, ny, nz, p_out_factor=0.995)
    lat, s = pair(fl, reaction=False)
    try:
        lat.Init()
        s.init()
        F = fluid(s)
        lat.calculate_moment()
        s.moments()
        for step in range(1, 3):
            s.collide_species(False)
            s.collide()
            s.stream()
            seed_gpu_from_oracle(lat, s)
            lat.TMS_BC()
            s.tms_bc()
            e = relerr(lat.get_populations(POP_F).reshape(9, 27, -1)[:, :, F], s.f[:, :, F])
            assert e < TOL, f"step {step} species f after TMS {e:.3e}"
            e = relerr(lat.get_populations(POP_G).reshape(27, -1)[:, F], s.g[:, F])
            assert e < TOL, f"step {step} g after TMS {e:.3e}"
            check_state(lat, s, TOL, f"step {step} after TMS")
            seed_gpu_from_oracle(lat, s)
            lat.calculate_moment()
            s.moments()
            check_state(lat, s, TOL, f"step {step}")
    finally:
        lat.close()
