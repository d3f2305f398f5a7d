"""Copies between host arrays and device layouts at the sizes where their form changes: 3 MB (several threads), 4 MB
slots, 64 MB passes; pageable and page-locked memory, unaligned and odd ones; and objects made and closed by several
threads at once, which share the kept slots and device blocks."""
import ctypes
import threading

import numpy as np
import pytest

import porelb_amd as P

pytestmark = pytest.mark.gpu

MB = 1 << 20


def lattice(nodes, **kw):
    side = int(np.ceil((nodes / 0.6) ** (1 / 3))) + 1
    flag = np.zeros(side ** 3, np.uint8)
    flag[np.random.default_rng(nodes).permutation(flag.size)[:nodes]] = 1
    kw = dict(dict(tau=0.8, gx=1e-5, bb_mode=P.BB_HALFWAY, index_kind=P.INDEX_TILE8, layout=P.LAYOUT_AOSOA,
                   ordering=P.ORDER_PENCIL, brick=(side, 8, 1), block_size=128), **kw)
    return P.Lattice.from_flag(flag.reshape(side, side, side), 1, **kw)


def state(lat, seed):
    rng = np.random.default_rng(seed)
    shape = lat.read_state().shape
    if lat.STATE_DTYPE[lat.cfg.precision] == np.uint16:
        return rng.integers(0, 0x3c00, shape).astype(np.uint16)
    w = 0.05 if lat.cfg.precision == P.FP64 else 0.0
    return (w + 1e-3 * rng.random(shape)).astype(lat.STATE_DTYPE[lat.cfg.precision])


# bytes of the state on either side of the threads' start, of a slot and of two, and of a long pass
@pytest.mark.parametrize("precision,nbytes", [
    (P.FP64, 152), (P.FP64, 3 * MB - 152), (P.FP64, 3 * MB + 152), (P.FP64, 4 * MB + 8), (P.FP64, 8 * MB + 304),
    (P.FP64, 65 * MB), (P.FP32, 3 * MB + 76), (P.FP32, 12 * MB + 76), (P.FP16, 3 * MB), (P.FP16, 9 * MB + 38)])
def test_state_both_ways(precision, nbytes):
    per = 19 * {P.FP64: 8, P.FP32: 4, P.FP16: 2}[precision]
    with lattice(max(1, nbytes // per), precision=precision) as lat:
        want = state(lat, 1)
        lat.write_state(want)
        assert np.array_equal(lat.read_state(), want)
        # the same through page-locked memory, and through pageable memory that is not aligned to a page or a line
        pinned = P.host_array(want.shape, want.dtype)
        pinned[...] = state(lat, 2)
        lat.write_state(pinned)
        raw = np.zeros(want.nbytes + 64, np.uint8)
        odd = raw[want.itemsize * 3:want.itemsize * 3 + want.nbytes].view(want.dtype).reshape(want.shape)
        rc = P.lib().plb_read_state(lat._h, ctypes.c_void_p(odd.ctypes.data))
        assert rc == 0 and np.array_equal(odd, pinned)
        lat.write_state(odd * 1)
        got = P.host_array(want.shape, want.dtype)
        rc = P.lib().plb_read_state(lat._h, ctypes.c_void_p(got.ctypes.data))
        assert rc == 0 and np.array_equal(got, odd)


@pytest.mark.parametrize("nodes", [1, 98_303, 98_305, 131_073, 262_145, 2_100_001])
def test_macros_components(nodes):
    with lattice(nodes, precision=P.FP32) as lat:
        lat.step(0, 3)
        want = lat.read_macros(P.host_array((4, lat.N)))
        assert np.array_equal(lat.read_macros(), want)
        assert np.array_equal(want[0] > 0.9, np.ones(lat.N, bool))
        # any subset of the four arrays
        for which in [(0,), (3,), (1, 2), (0, 1, 3)]:
            out = np.full((4, lat.N), np.nan)
            args = [ctypes.c_void_p(out[q].ctypes.data) if q in which else None for q in range(4)]
            assert P.lib().plb_read_macros(lat._h, *args) == 0
            for q in range(4):
                assert np.array_equal(out[q], want[q]) if q in which else np.isnan(out[q]).all()


def test_records_of_a_large_mask():
    flag = (np.random.default_rng(0).random((90, 91, 93)) < 0.5).astype(np.uint8)
    V, start = P.preprocess(flag, 3)
    N = int(flag.sum())
    assert len(V) == N and start[0] == 0   # 58 MB of records: several slots
    small = P.preprocess(flag[:30], 1)[0]  # 19 MB
    z, y, x = np.nonzero(flag)
    key = (V["z"].astype(np.int64) * 91 + V["y"]) * 93 + V["x"]
    assert np.array_equal(np.sort(key), (z * 91 + y) * 93 + x)
    assert len(small) == int(flag[:30].sum())
    # the records of the first slab do not depend on what comes after it, but for the links over its faces
    same = small["z"] % 29 != 0
    assert np.array_equal(small[["x", "y", "z"]], V[:len(small)][["x", "y", "z"]])
    assert np.array_equal(small["nb"]["node_id"][same], V[:len(small)]["nb"]["node_id"][same])


def test_threads_share_slots_and_blocks():
    def work(k, out):
        rows = []
        for rep in range(3):
            with lattice(60_000 + 40_000 * k + rep, precision=P.FP64) as lat:
                s = state(lat, k)
                lat.write_state(s)
                lat.step(0, 4)
                rows.append((lat.read_state(), lat.read_macros()))
        out[k] = rows

    alone, shared = [None] * 6, [None] * 6
    for k in range(6):
        work(k, alone)
    threads = [threading.Thread(target=work, args=(k, shared)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, shared):
        for (s0, m0), (s1, m1) in zip(a, b):
            assert np.array_equal(s0, s1) and np.array_equal(m0, m1)


# 8 365 427 and 8 406 636 voxels: 130 710 and 131 354 words of the mask, either side of the one-block scan's 131 072
@pytest.mark.parametrize("nx", [203, 204])
def test_order_and_table_of_large_masks(nx):
    flag = (np.random.default_rng(nx).random((203, 203, nx)) < 0.06).astype(np.uint8)
    out = []
    for kw in (dict(), dict(index_kind=P.INDEX_TILE8, layout=P.LAYOUT_AOSOA, ordering=P.ORDER_PENCIL,
                            brick=(nx, 64, 1), block_size=128)):
        with P.Lattice.from_flag(flag, 1, tau=0.8, gx=1e-5, precision=P.FP64, bb_mode=P.BB_HALFWAY, **kw) as lat:
            table = lat.read_table()
            lat.step(0, 5)
            out.append((table, lat.read_state()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("managed", [False, True])
@pytest.mark.parametrize("nbytes", [1 * MB, 3 * MB + 152, 20 * MB])
def test_device_and_managed_memory(nbytes, managed):
    """Arrays that are not host memory, on both sides of the size from which threads move host memory."""
    L = P.lib()
    hip = ctypes.CDLL("libamdhip64.so")     # the one libplb.so has loaded
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    with lattice(nbytes // 152, precision=P.FP64) as lat:
        want = state(lat, 5)
        p, size = ctypes.c_void_p(), ctypes.c_size_t(want.nbytes)
        assert (hip.hipMallocManaged(ctypes.byref(p), size, 1) if managed else hip.hipMalloc(ctypes.byref(p), size)) == 0

        def back(n):
            out = np.zeros(n)
            assert hip.hipMemcpy(out.ctypes.data, p, out.nbytes, 4) == 0
            return out

        lat.write_state(want)
        assert L.plb_read_state(lat._h, p) == 0
        assert np.array_equal(back(want.size).reshape(want.shape), want)
        lat.init_equilibrium()
        assert L.plb_write_state(lat._h, p) == 0
        assert np.array_equal(lat.read_state(), want)
        lat.step(0, 3)
        assert L.plb_read_populations(lat._h, p) == 0
        assert np.array_equal(back(want.size).reshape(want.shape), lat.read_populations())
        macros = lat.read_macros()
        parts = [ctypes.c_void_p(p.value + 8 * lat.N * q) for q in range(4)]
        assert L.plb_read_macros(lat._h, *parts) == 0
        assert np.array_equal(back(4 * lat.N).reshape(4, lat.N), macros)
        hip.hipFree(p)


def test_some_arrays_page_locked():
    with lattice(300_000, precision=P.FP32) as lat:
        lat.step(0, 3)
        want = lat.read_macros()
        out = [np.zeros(lat.N), P.host_array(lat.N), np.zeros(lat.N), P.host_array(lat.N)]
        assert P.lib().plb_read_macros(lat._h, *[ctypes.c_void_p(o.ctypes.data) for o in out]) == 0
        assert all(np.array_equal(o, w) for o, w in zip(out, want))


def test_release_memory():
    """Device blocks that stay after the last lattice go back to the system on request."""
    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    def use():
        with lattice(200_000, precision=P.FP32) as lat:
            lat.step(0, 200)
            return lat.read_state()

    want = use()
    P.release_memory()
    before = free()
    assert np.array_equal(use(), want)
    assert free() < before - 16 * MB      # kept for the next one
    P.release_memory()
    assert free() >= before - 4 * MB
    assert np.array_equal(use(), want)


def test_bricks_past_the_mask_make_more_than_2_32_voxels():
    """1620^3 voxels are less than 2^32, rows of 64 rounded up (1664) make more."""
    edge = 1620
    flag = np.zeros((edge, edge, edge), np.uint8)
    rng = np.random.default_rng(8)
    for z, y, x in [(0, 0, 0), (edge - 20, edge - 20, edge - 40), (800, 1590, 700), (edge - 20, 0, 0)]:
        flag[z:z + 20, y:y + 20, x:x + 40] = rng.random((20, 20, 40)) < 0.8
    out = []
    for kw in (dict(ordering=P.ORDER_REFERENCE), dict(ordering=P.ORDER_PENCIL, brick=(edge, 64, 1))):
        with P.Lattice.from_flag(flag, 1, tau=0.8, gx=1e-5, precision=P.FP64, bb_mode=P.BB_HALFWAY, **kw) as lat:
            table = lat.read_table()
            lat.step(0, 9)
            out.append((table, lat.read_state()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
