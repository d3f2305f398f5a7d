"""On-chip runs that cannot complete: a launch without its last block, as when
that block finds no room on the chip.  The other blocks' waits end, and the run
is repeated with one launch per step, with the results of that."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE = dict(index_kind=1, layout=1, ordering=2, block_size=128)


def withhold(plb, obj, runs):
    """The next `runs` launches go without a block; returns how many were still to come."""
    name = "plb_test_batch_withhold_block" if isinstance(obj, plb.Batch) else "plb_test_withhold_block"
    f = getattr(plb.lib(), name)
    f.argtypes, f.restype = [C.c_void_p, C.c_int], C.c_int
    return f(obj._h, runs)


def same(a, b):
    assert np.array_equal(a.read_state(), b.read_state())
    assert np.array_equal(a.read_macros(), b.read_macros())


def pair(plb, precision, tau=0.8, gx=1e-5):
    flag = plb.mask_spheres((30, 32, 34), 3.0, 5.0, 0.5, 4)
    kw = dict(tau=tau, gx=gx, precision=precision, bb_mode=1, fp16_rounding=1, brick=(34, 8, 1), **SHAPE)
    return plb.Lattice.from_flag(flag, **kw), plb.Lattice.from_flag(flag, graph_steps=1024, **kw)


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_queue_with_a_run_that_gives_up(plb, precision):
    a, b = pair(plb, precision)
    L = plb.lib()
    with a, b:
        for lat in (a, b):
            lat.step(0, 130)
        assert L.plb_step_async(a._h, 130, 41) == 0
        withhold(plb, a, 1)
        for call in [(171, 40), (211, 33), (244, 7)]:
            assert L.plb_step_async(a._h, *call) == 0
        assert withhold(plb, a, 0) == 0
        assert L.plb_sync(a._h) == 0
        for call in [(130, 41), (171, 40), (211, 33), (244, 7)]:
            b.step(*call)
        same(a, b)


def test_trip_in_a_run_that_gives_up(plb):
    a, b = pair(plb, 0, 0.51, 0.003)
    with a, b:
        a.step_rc(0, 130)
        a.init_equilibrium()
        withhold(plb, a, 1)
        assert a.step_rc(0, 130) == b.step_rc(0, 130) == plb.ERR_DENSITY
        assert a.last_fault() == b.last_fault()
        same(a, b)


def batch(plb, precision, gx=1e-5):
    flags = [plb.mask_spheres((30, 32, 34), 3.0, 5.0, 0.5, 4 + k) for k in range(3)]
    kw = dict(precision=precision, bb_mode=1, fp16_rounding=1, brick=(34, 8, 1), **SHAPE)
    taus, gxs = [0.8, 0.51, 0.9], [1e-5, gx, 2e-5]
    return plb.Batch(flags, taus, gxs, **kw), plb.Batch(flags, taus, gxs, **kw)


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_batch_that_gives_up(plb, precision):
    a, b = batch(plb, precision)
    withhold(plb, a, 5)
    ra, rb = a.run(150, 50, 0.0), b.run(150, 15, 0.0)
    assert withhold(plb, a, 5) == 4        # one launch gave up, and the run was not tried on chip again
    assert np.array_equal(ra[0], rb[0]) and ra[1] == rb[1]
    for s in range(3):
        assert np.array_equal(a.read_macros(s), b.read_macros(s))
    assert a.reduce() == b.reduce()
    a.run(150, 50, 0.0)
    assert withhold(plb, a, 0) == 5        # nor was the next one
    a.close()
    b.close()


def test_batch_that_gives_up_and_trips(plb):
    """The density guard trips in the launch that gives up: it still counts as one."""
    a, b = batch(plb, 0, 0.03)
    withhold(plb, a, 5)
    for x, every in ((a, 50), (b, 10)):
        with pytest.raises(plb.PlbError) as e:
            x.run(150, every, 0.0)
        assert e.value.code == plb.ERR_DENSITY
    assert a.last_fault() == b.last_fault() and a.last_fault()[0] == 1
    assert withhold(plb, a, 5) == 4
    with pytest.raises(plb.PlbError):
        a.run(150, 50, 0.0)
    assert withhold(plb, a, 0) == 5
    a.close()
    b.close()


def test_chip_is_tried_again(plb):
    """After a run that gave up, 16 384 steps with one launch each and then the chip
    again; after the next one, twice as many."""
    a, b = pair(plb, 1)
    with a, b:
        it = 0

        def steps(n, call=512):
            nonlocal it
            for end in range(it + call, it + n + 1, call):
                a.step(it, call)
                it = end

        steps(160, 160)
        for pause in (16384, 32768):
            withhold(plb, a, 1)
            steps(64, 64)
            assert withhold(plb, a, 1) == 0      # gave up
            steps(pause)
            assert withhold(plb, a, 0) == 1      # none on chip
        steps(96, 96)
        for s in range(0, it, 1000):
            b.step(s, min(1000, it - s))
        same(a, b)


def test_batch_is_tried_again(plb):
    a, b = batch(plb, 1)
    withhold(plb, a, 5)
    a.run(150, 50, 0.0)
    withhold(plb, a, 5)
    a.run(16384, 1000, 0.0)
    assert withhold(plb, a, 5) == 5
    a.run(150, 50, 0.0)
    assert withhold(plb, a, 0) == 4
    b.run(150, 15, 0.0)
    assert a.reduce() == b.reduce()
    a.close()
    b.close()


def test_lattices_on_chip_at_the_same_time(plb):
    """Three threads with a lattice that fills the chip each, and a fourth with one
    that does not fit it: whatever of them gives up, the results are those of each alone."""
    flags = [plb.mask_noise((64, 64, 64), 2.0, 0.35, k) for k in range(3)] + [plb.mask_noise((128, 128, 128), 2.0, 0.4, 9)]

    def work(k):
        kw = dict(tau=0.8, gx=1e-5, precision=k % 2, bb_mode=1, brick=(flags[k].shape[2], 8, 1), **SHAPE)
        with plb.Lattice.from_flag(flags[k], **kw) as lat:
            for it in range(0, 2000, 200):
                lat.step(it, 200)
            return lat.read_state(), lat.read_macros()

    alone, shared = [work(k) for k in range(4)], [None] * 4
    threads = [threading.Thread(target=lambda k=k: shared.__setitem__(k, work(k))) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for one, other in zip(alone, shared):
        assert np.array_equal(one[0], other[0]) and np.array_equal(one[1], other[1])


def test_time_of_repeated_steps(plb):
    """plb_step_timed gives the time of the steps, not that of the run that gave up."""
    a, b = pair(plb, 0)
    with a, b:
        a.step(0, 130)
        b.step(0, 130)
        n = 40_000
        want = b.step_timed(130, n)
        assert want > 80.0
        withhold(plb, a, 1)
        ms = a.step_timed(130, n)
        assert withhold(plb, a, 0) == 0
        assert 0.5 * want < ms < 2.0 * want
        same(a, b)


def test_time_of_the_call_that_builds_the_plan(plb):
    """The plan of the on-chip runs is not in the time of the first one."""
    first, later = [], []
    for _ in range(6):
        a, b = pair(plb, 0)
        with a, b:
            first.append(a.step_timed(0, 200))
            later.append(a.step_timed(200, 200))
    assert min(first) < 1.4 * min(later)
