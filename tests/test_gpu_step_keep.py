"""Step kernels with plain and with non-temporal stores compute the same: lattices on both sides of the sizes
(32, 208 and 600 MB of populations and index) between which all or some blocks store plainly, against the
two-nodes-per-thread kernel, which has non-temporal stores."""
import numpy as np
import pytest

import porelb_amd as P

pytestmark = pytest.mark.gpu


# pore nodes x (2 x 19 x element + index bytes): FP64 with an int32 table 376 bytes a node, FP32 224
@pytest.mark.parametrize("layout", [P.LAYOUT_SOA, P.LAYOUT_AOSOA])
@pytest.mark.parametrize("precision,bb,nodes", [
    (P.FP64, P.BB_REFCOMPAT, 85_000), (P.FP64, P.BB_REFCOMPAT, 85_207), (P.FP64, P.BB_HALFWAY, 553_100),
    (P.FP64, P.BB_HALFWAY, 553_299), (P.FP64, P.BB_HALFWAY, 1_595_700), (P.FP64, P.BB_HALFWAY, 1_595_800),
    (P.FP32, P.BB_HALFWAY, 142_000), (P.FP32, P.BB_REFCOMPAT, 142_931), (P.FP32, P.BB_HALFWAY, 1_200_001)])
def test_same_as_two_nodes_per_thread(precision, bb, nodes, layout):
    rng = np.random.default_rng(nodes)
    flag = np.zeros(120 * 121 * 119, np.uint8)
    flag[rng.permutation(flag.size)[:nodes]] = 1
    flag = flag.reshape(119, 121, 120)
    out = []
    for per_thread in (1, 2):
        with P.Lattice.from_flag(flag, 1, tau=0.8, gx=1e-5, precision=precision, bb_mode=bb, layout=layout,
                                 nodes_per_thread=per_thread) as lat:
            lat.step(0, 7)
            lat.step(7, 4)
            out.append((lat.read_state(), lat.read_macros()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("index", [P.INDEX_I32, P.INDEX_TILE8, P.INDEX_BITMAP])
def test_index_kinds(index):
    flag = (np.random.default_rng(3).random((60, 70, 80)) < 0.5).astype(np.uint8)
    out = []
    for per_thread in (1, 2):
        with P.Lattice.from_flag(flag, 1, tau=0.8, gx=1e-5, precision=P.FP64, bb_mode=P.BB_HALFWAY, index_kind=index,
                                 layout=P.LAYOUT_AOSOA, nodes_per_thread=per_thread) as lat:
            lat.step(0, 9)
            out.append((lat.read_state(), lat.read_macros()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
