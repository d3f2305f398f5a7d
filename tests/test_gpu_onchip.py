"""On-chip runs (calls of 16 steps or more of a lattice whose populations fit
the LDS) against calls of 15 steps, which take one launch per step: stored
state and macros bit for bit, at the edges of the block sizes, in both bounce
modes, over odd extents, through a density-guard trip, and for V records that
no mask gives, which must stay off the on-chip path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CUS = 256
SHAPE = dict(index_kind=1, layout=1, ordering=2)


def mask_of(n, shape, seed):
    """A random mask with exactly n pores."""
    m = np.zeros(int(np.prod(shape)), dtype=np.uint8)
    m[np.random.default_rng(seed).permutation(m.size)[:n]] = 1
    return m.reshape(shape)


def same(a, b, calls):
    """Advances a by whole calls and b by calls of at most 15 steps."""
    it = 0
    for n in calls:
        a.step(it, n)
        for s in range(0, n, 15):
            b.step(it + s, min(15, n - s))
        it += n
        assert np.array_equal(a.read_state(), b.read_state())
        assert np.array_equal(a.read_macros(), b.read_macros())


# (precision, nodes): one block; a full and an overfull slot count of each
# kernel variant (2 or 1 copies in LDS, 1 or 2 nodes per thread); the largest
# lattice that fits and the first that does not.
EDGES = [(p, n) for p in (0, 1, 2) for n in (1, 255, 257, 256 * CUS, 256 * CUS + 1)] + [
    (0, 512 * CUS), (0, 512 * CUS + 1), (0, 1024 * CUS), (0, 1024 * CUS + 1),
    (1, 1024 * CUS), (1, 1024 * CUS + 1), (1, 2048 * CUS), (1, 2048 * CUS + 1),
    (2, 1024 * CUS), (2, 1024 * CUS + 1), (2, 2048 * CUS), (2, 2048 * CUS + 1)]


@pytest.mark.parametrize("precision,nodes", EDGES)
def test_block_sizes(plb, precision, nodes):
    edge = max(4, int(np.ceil((nodes / 0.6) ** (1 / 3))))
    flag = mask_of(nodes, (edge, edge + 1, edge + 2), nodes)
    kw = dict(tau=0.8, gx=1e-5, precision=precision, bb_mode=nodes % 2, fp16_rounding=1, brick=(edge + 2, 16, 1), **SHAPE)
    with plb.Lattice.from_flag(flag, **kw) as a, plb.Lattice.from_flag(flag, **kw) as b:
        same(a, b, [130, 17])


@pytest.mark.parametrize("index,layout,order", [(0, 0, 0), (0, 1, 1), (1, 0, 2), (2, 1, 2), (2, 0, 0)])
@pytest.mark.parametrize("dims", [(1, 1, 70), (2, 3, 64), (37, 5, 41), (31, 33, 30)])
def test_shapes_and_extents(plb, dims, index, layout, order):
    flag = mask_of(max(1, int(0.7 * np.prod(dims))), dims, 3)
    brick = (dims[2], 4, 1) if order == 2 else (8, 4, 2)
    kw = dict(tau=0.7, gx=2e-5, precision=1, bb_mode=1, index_kind=index, layout=layout, ordering=order, brick=brick)
    with plb.Lattice.from_flag(flag, **kw) as a, plb.Lattice.from_flag(flag, **kw) as b:
        same(a, b, [128, 16, 33])


@pytest.mark.parametrize("ranks", [1, 3])
def test_reference_order_against_oracle(plb, oracle_mod, ranks):
    O = oracle_mod
    flag = mask_of(9000, (24, 26, 28), 9)
    V, start = O.build_V(flag, ranks)
    f0, _ = O.init_equilibrium(len(V))
    mac = O.pull_run(O.pull_table(V, start, O.BB_REFCOMPAT), f0, 150, 0.8, 1e-4)
    with plb.Lattice.from_flag(flag, ranks, tau=0.8, gx=1e-4, brick=(28, 8, 1), **SHAPE) as lat:
        lat.step(0, 150)
        assert np.array_equal(lat.read_populations(), f0)
        assert np.array_equal(lat.read_macros(), mac)


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_density_guard_trip(plb, precision):
    """The trip falls inside an on-chip run, with another call queued behind it."""
    flag = mask_of(15000, (30, 32, 34), 4)
    kw = dict(tau=0.51, gx=0.03, precision=precision, bb_mode=1, brick=(34, 8, 1), **SHAPE)
    L = plb.lib()
    with plb.Lattice.from_flag(flag, **kw) as a, plb.Lattice.from_flag(flag, **kw) as b:
        assert b.step_rc(0, 15) == plb.ERR_DENSITY
        fault = b.last_fault()
        assert 5 <= fault["step"] < 15
        assert L.plb_step_async(a._h, 0, 400) == 0
        assert L.plb_step_async(a._h, 400, 100) == 0
        assert L.plb_sync(a._h) == plb.ERR_DENSITY
        assert a.last_fault() == fault
        assert np.array_equal(a.read_state(), b.read_state())
        assert np.array_equal(a.read_macros(), b.read_macros())
        assert a.step_rc(500, 200) == plb.ERR_DENSITY      # still frozen
        assert np.array_equal(a.read_state(), b.read_state())
        # queued, read without a plb_sync
        a.init_equilibrium()
        assert L.plb_step_async(a._h, 0, 200) == 0
        assert a.last_fault() == fault
        assert np.array_equal(a.read_macros(), b.read_macros())
        assert L.plb_sync(a._h) == plb.ERR_DENSITY
        assert np.array_equal(a.read_state(), b.read_state())


@pytest.mark.parametrize("what", ["link", "coordinates"])
def test_records_that_contradict_each_other(plb, what):
    """plb_create takes V records as they are; a link whose other end points
    elsewhere, or two nodes on one voxel, still step as one launch per step does."""
    flag = mask_of(3000, (16, 18, 20), 6)
    V, start = plb.preprocess(flag, 1)
    V = V.copy()
    if what == "link":
        k = int(np.flatnonzero(V["nb"]["node_type"][:, 0] == plb.TYPE_FLUID)[5])
        V["nb"]["node_id"][k, 0] = (int(V["nb"]["node_id"][k, 0]) + 1500) % len(V)
    else:
        for c in "xyz":
            V[c][10] = V[c][2000]
    kw = dict(tau=0.8, gx=1e-5, bb_mode=1)
    with plb.Lattice.from_V(V, start, flag.shape, **kw) as a, plb.Lattice.from_V(V, start, flag.shape, **kw) as b:
        same(a, b, [130, 20])


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("persistent", [False, True])
def test_batch_on_chip(plb, precision, persistent):
    """Samples on chip (checks 16 steps or more apart) against launches per step
    (checks 15 apart): macros bit for bit; one sample has no pores, one does not
    fit the chip in FP64, and the samples take more than one launch."""
    rng = np.random.default_rng(12)
    flags = [mask_of(int(0.55 * np.prod(d)), d, k) for k, d in
             enumerate([(20, 21, 22), (64, 62, 60), (9, 70, 8), (80, 78, 81), (30, 30, 30)])]
    flags.insert(2, np.zeros((5, 5, 5), np.uint8))
    taus = [0.6 + 0.1 * k for k in range(6)]
    gxs = [10.0 ** -(5 + 0.2 * k) for k in range(6)]
    kw = dict(precision=precision, bb_mode=1, fp16_rounding=1, block_size=128, brick=(1, 16, 1), **SHAPE)
    a, b = plb.Batch(flags, taus, gxs, **kw), plb.Batch(flags, taus, gxs, **kw)
    for every, steps in ((50, 150), (33, 145)):
        ra = a.run(steps, every, 0.0, persistent=persistent)
        rb = b.run(steps, 15, 0.0)
        assert np.array_equal(ra[0], rb[0]) and ra[1] == rb[1]
        assert all(np.array_equal(a.read_macros(s), b.read_macros(s)) for s in range(6))
        assert a.reduce() == b.reduce()
    a.close()
    b.close()


def test_batch_stops_and_trips(plb):
    """Samples that stop at their own steps, as single lattices do; and a
    density-guard trip, which ends as it does with one launch per step."""
    flags = [mask_of(4000 + 900 * k, (20, 22, 24), 20 + k) for k in range(4)]
    kw = dict(precision=0, bb_mode=1, block_size=128, brick=(24, 8, 1), **SHAPE)
    taus, gxs = [0.7, 0.8, 1.0, 1.2], [1e-5, 2e-5, 1e-6, 3e-6]
    b = plb.Batch(flags, taus, gxs, **kw)
    steps, _, _ = b.run(2000, 20, 1e-3)
    assert 0 < steps.min() < steps.max() < 2000
    for s in range(4):
        with plb.Lattice.from_flag(flags[s], tau=taus[s], gx=gxs[s], **kw) as lat:
            n, r = lat.run_to_convergence(0, 2000, 20, 1e-3)
            assert n == steps[s] and np.array_equal(lat.read_macros(), b.read_macros(s))
    b.close()
    gxs[2] = 0.05
    taus[2] = 0.51
    a, b = plb.Batch(flags, taus, gxs, **kw), plb.Batch(flags, taus, gxs, **kw)
    for x, every in ((a, 50), (b, 10)):
        with pytest.raises(plb.PlbError) as e:
            x.run(200, every, 0.0)
        assert e.value.code == plb.ERR_DENSITY
    assert a.last_fault() == b.last_fault() and a.last_fault()[0] == 2
    a.close()
    b.close()


@pytest.mark.parametrize("large", [0, 1, 3])
def test_batch_with_a_sample_off_chip(plb, large):
    """Samples on chip before, between and behind one that is too large for it:
    the plan numbers its own samples' nodes only."""
    flags = [mask_of(n, d, k) for k, (n, d) in enumerate([(3000, (20, 21, 22)), (40001, (41, 42, 43)), (700, (9, 70, 8))])]
    flags.insert(large, mask_of(560_003, (100, 101, 102), 7))
    taus, gxs = [0.6 + 0.1 * k for k in range(4)], [10.0 ** -(5 + 0.2 * k) for k in range(4)]
    kw = dict(precision=1, bb_mode=large % 2, block_size=128, brick=(1, 16, 1), **SHAPE)
    a, b = plb.Batch(flags, taus, gxs, **kw), plb.Batch(flags, taus, gxs, **kw)
    ra, rb = a.run(140, 70, 0.0), b.run(140, 14, 0.0)
    assert np.array_equal(ra[0], rb[0]) and ra[1] == rb[1]
    assert all(np.array_equal(a.read_macros(s), b.read_macros(s)) for s in range(4))
    assert a.reduce() == b.reduce()
    a.close()
    b.close()
