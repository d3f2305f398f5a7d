"""Density-guard trips in queues of asynchronous calls: the fault, the frozen
state and the macros are those of the same calls made one by one with one
launch per step (graph_steps longer than any call keeps a lattice to that)."""
import pytest

import numpy as np

pytestmark = pytest.mark.gpu

# Without the guard's trip the flow would be past it at about step 46 (FP64, counted from rest).
GX = 0.003


def pair(plb, precision, gx=GX):
    flag = plb.mask_spheres((30, 32, 34), 3.0, 5.0, 0.5, 4)
    kw = dict(tau=0.51, gx=gx, precision=precision, bb_mode=1, fp16_rounding=1, index_kind=1, layout=1, ordering=2,
              brick=(34, 8, 1), block_size=128)
    return plb.Lattice.from_flag(flag, **kw), plb.Lattice.from_flag(flag, graph_steps=1024, **kw)


def warm(lat):
    """Past the 128 steps from which calls of 16 or more run on chip."""
    lat.step_rc(0, 130)
    lat.init_equilibrium()


def one_by_one(plb, lat, calls):
    """The calls, each waited for, up to the first that trips."""
    for it0, n in calls:
        rc = lat.step_rc(it0, n)
        if rc:
            return rc
    return 0


def same(a, b):
    assert a.last_fault() == b.last_fault()
    assert np.array_equal(a.read_state(), b.read_state())
    assert np.array_equal(a.read_macros(), b.read_macros())


@pytest.mark.parametrize("read", ["", "read", "reduce"])
@pytest.mark.parametrize("n", [60, 61, 30, 31])   # the trip falls into the first call, into the second
@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("chip", [True, False])
def test_step_numbers_that_start_again(plb, chip, precision, n, read):
    a, b = pair(plb, precision)
    if not chip:
        a = pair(plb, precision)[1]
    L = plb.lib()
    with a, b:
        if chip:
            warm(a)
        rc = one_by_one(plb, b, [(0, n), (0, n)])
        assert rc == plb.ERR_DENSITY
        assert L.plb_step_async(a._h, 0, n) == 0
        if read:
            a.read_macros() if read == "read" else a.reduce()
        assert L.plb_step_async(a._h, 0, n) == 0
        assert L.plb_sync(a._h) == rc
        same(a, b)
        # and from rest again, on chip as before
        a.init_equilibrium()
        b.init_equilibrium()
        assert a.step_rc(0, n) == b.step_rc(0, n)
        same(a, b)


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_trip_in_front_of_a_queued_run(plb, precision):
    """The trip falls into launches per step, before the 128th step; the call
    queued behind them would run on chip, and is held off."""
    a, b = pair(plb, precision)
    L = plb.lib()
    with a, b:
        rc = one_by_one(plb, b, [(0, 100), (100, 100)])
        assert rc == plb.ERR_DENSITY
        assert L.plb_step_async(a._h, 0, 100) == 0
        assert L.plb_step_async(a._h, 100, 100) == 0
        assert L.plb_sync(a._h) == rc
        same(a, b)


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_queued_runs_before_a_trip_and_behind_it(plb, precision):
    """On-chip runs by turns with short calls; the trip falls into a short one."""
    a, b = pair(plb, precision)
    L = plb.lib()
    with a, b:
        warm(a)
        b.step_rc(0, 200)
        trip = b.last_fault()["step"]
        b.init_equilibrium()
        calls = [(0, trip - 5), (trip - 5, 12), (trip + 7, 40), (trip + 47, 3)]
        rc = one_by_one(plb, b, calls)
        assert rc == plb.ERR_DENSITY and b.last_fault()["step"] == trip
        for it0, n in calls:
            assert L.plb_step_async(a._h, it0, n) == 0
        assert a.last_fault() == b.last_fault()     # a read before plb_sync
        assert np.array_equal(a.read_macros(), b.read_macros())
        assert L.plb_step_async(a._h, trip + 100, 60) == 0
        assert L.plb_sync(a._h) == rc
        same(a, b)


@pytest.mark.parametrize("gap", [0, 1])
def test_queue_without_a_sync_stays_small(plb, gap):
    """Asynchronous calls and reads, never a plb_sync: no memory for every call."""
    def resident():
        return int(open("/proc/self/statm").read().split()[1]) * 4096

    L = plb.lib()
    a, b = pair(plb, 1, gx=1e-6)
    with a, b:
        it = 0

        def queue(calls):
            nonlocal it
            for k in range(calls):
                assert L.plb_step_async(b._h, it, 1) == 0
                it += 1 + gap
                if k % 1000 == 0:
                    b.reduce()

        queue(20_000)
        before = resident()
        queue(400_000)
        assert resident() - before < 4 << 20
        assert L.plb_sync(b._h) == 0


def test_long_queue_ends_in_the_same_state(plb):
    """More calls than the queue holds, on chip and between, and a trip behind them."""
    a, b = pair(plb, 0, gx=0.002)     # trips at about step 144
    L = plb.lib()
    with a, b:
        warm(a)
        # steps in a row, steps with gaps in their numbers, on-chip runs
        calls = [(k, 1) for k in range(140)] + [(140 + 2 * k, 1) for k in range(300)] + [(800, 20), (820, 20), (840, 3)]
        rc = one_by_one(plb, b, calls)
        for it0, n in calls:
            assert L.plb_step_async(a._h, it0, n) == 0
        assert L.plb_sync(a._h) == rc == plb.ERR_DENSITY
        same(a, b)


@pytest.mark.parametrize("frozen", [65_530, 65_531])
def test_runs_after_a_long_held_off_call(plb, frozen):
    """FP16 words carry 16 bits of the step number, which a held-off call of this
    length brings round to those that the run before it left in the buffers."""
    a, b = pair(plb, 2)
    good = plb.Lattice.from_flag(plb.mask_spheres((30, 32, 34), 3.0, 5.0, 0.5, 4), tau=0.51, gx=GX, precision=2, bb_mode=1)
    L = plb.lib()
    with a, b, good:
        warm(a)
        good.step(0, 20)
        state = good.read_state()
        for call in [(0, 200), (200, frozen)]:
            assert L.plb_step_async(a._h, *call) == 0
        assert L.plb_sync(a._h) == plb.ERR_DENSITY
        a.write_state(state)
        b.write_state(state)
        assert a.step_rc(0, 20) == b.step_rc(0, 20)
        same(a, b)
