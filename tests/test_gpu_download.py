"""Large downloads (through the pinned staging) against small ones of the same values.

A grid whose field planes pass the staging threshold is filled with a value
per cell and read back whole: fields (binary64), populations (binary32 storage
with its per-plane shifts), species planes (binary64, and binary32 without a
shift below and above the threshold), lengths that are no multiple of the chunk,
twice over and from two threads with a context each."""
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from lbm_amd import cases
from lbm_amd.capi import LBM_FP32_SHIFTED, LBM_FP64, LBM_MODE_STRICT, POP_F, POP_G, Lattice, MixtureLattice


def _values(shape, seed):
    return np.random.default_rng(seed).random(shape)


@pytest.mark.parametrize("shape", [(126, 127, 131), (127, 130, 125)])  # 17.57 and 17.30 MB planes, odd lengths
def test_fields_come_back(shape):
    lat = Lattice(*shape, 0.1, mode=LBM_MODE_STRICT)
    for rep in range(2):
        for k, name in enumerate(("rho", "T", "HRR")):
            a = _values(lat.shape, 10 * rep + k)
            lat.set_field(name, a)
            assert np.array_equal(lat.get_field(name), a)
    lat.close()


@pytest.mark.parametrize("precision", [LBM_FP64, LBM_FP32_SHIFTED])
def test_species_planes_and_populations_come_back(precision):
    n = (62, 53, 70)
    lat = MixtureLattice(*n, *cases.UNITS_FLAME, precision=precision, mode=LBM_MODE_STRICT)
    fl = cases.reacting_box(*n, X={s: 1.0 for s in cases.H2AIR_SPECIES})
    lat.load_case(fl)
    lat.Init()
    X = _values((9,) + lat.shape, 5).astype(np.float32).astype(np.float64)
    lat.set_species_field("X", X)
    got = lat.get_species_field("X")
    assert np.array_equal(got, X)
    # populations: what is uploaded comes back, in FP32 to the storage's rounding
    for which, shape in ((POP_F, (9, 27) + lat.shape), (POP_G, (27,) + lat.shape)):
        f = 0.01 * _values(shape, 6)
        lat.set_populations(which, f)
        a = lat.get_populations(which)
        if precision == LBM_FP64:
            assert np.array_equal(a, f)
        else:
            # value - shift in binary32: half a unit in the last place of |f| + |shift| <= 1
            assert np.max(np.abs(a - f)) <= 2.0 ** -24
    lat.close()


def test_binary32_species_planes_come_back():
    n = (100, 91, 90)  # nine planes of 102 x 93 x 92 binary32 values: 31.4 MB
    lat = MixtureLattice(*n, *cases.UNITS_FLAME, precision=LBM_FP32_SHIFTED, mode=LBM_MODE_STRICT)
    for k, name in enumerate(("X", "u")):
        a = _values((9,) + lat.shape, 8 + k).astype(np.float32).astype(np.float64)
        lat.set_species_field(name, a)
        assert np.array_equal(lat.get_species_field(name), a)
    lat.close()


def test_two_threads_download_at_once():
    errs = []

    def one(seed):
        try:
            lat = Lattice(126, 127, 131, 0.1, mode=LBM_MODE_STRICT)
            a = _values(lat.shape, seed)
            lat.set_field("p", a)
            for _ in range(3):
                if not np.array_equal(lat.get_field("p"), a):
                    errs.append(seed)
            lat.close()
        except Exception as e:  # noqa: BLE001
            errs.append(repr(e))

    ts = [threading.Thread(target=one, args=(s,)) for s in (1, 2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not errs


def test_waiting_for_queued_steps_takes_one_thread():
    """A field read after queued steps: the wait for them is one thread's, the copying
    threads start after it.  So the read takes the processor time of the same read
    without queued steps and, at most, the wait's twice over (the waiting thread may
    spin, and the runtime has a thread of its own); eight waiting threads take more."""
    lat = Lattice(256, 256, 256, 0.1, precision=LBM_FP32_SHIFTED)
    fl = cases.default_fields(256, 256, 256)
    cases.periodic_ghosts(fl)
    fl["p"][...], fl["T"][...] = 1.0 / 3.0, 1.0
    lat.load_case(fl)
    lat.Init()

    def read():
        wall, cpu = time.perf_counter(), time.process_time()
        lat.get_field("T")
        return time.perf_counter() - wall, time.process_time() - cpu

    lat.step(3)
    lat.get_field("T")
    lat.sync()
    _, idle = read()
    lat.step(80)
    wall, cpu = read()
    lat.close()
    assert cpu - idle < 2 * wall, (wall, cpu, idle)
