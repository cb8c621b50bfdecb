"""Distances over whole lengths whose first long list, which the host enqueues a round for before it knows the lengths, has one edge a lane, just
short of two chunks a work-group, or eight edges a lane: against the oracle, exactly (sums of whole numbers)."""
import numpy as np
import pytest

from test_traverse_rounds_gpu import _layers

pytestmark = pytest.mark.gpu

# out-edges of the second list: 128 work-groups of 256 lanes have a chunk each up to 32,768, two up to 65,535
WIDTHS = {"one": (8_192, 4), "two": (16_383, 4), "wide": (16_384, 4), "wide_more": (16_385, 4), "long": (60_000, 3), "tail": (20_001, 5)}


@pytest.mark.parametrize("name", WIDTHS)
def test_first_long_list(oracle, name):
    from drone_amd.traverse import SSSPWorkerCUDA
    width, fan = WIDTHS[name]
    u, v = _layers([1, 3000, width, 40_000, 70, 3], fan, 11)
    nglobal = int(max(u.max(), v.max())) + 1
    n, g2l, l2g, index, dst = oracle.build_graph(nglobal, u, v)
    length = np.random.default_rng(width).integers(1, 9, len(dst)).astype(np.float32)
    st = oracle.SSSPState(index, dst, length)
    st.peval(int(g2l[0]))
    w = SSSPWorkerCUDA(nglobal, u, v, startId=0)
    try:
        w.set_edge_len(length)
        for _ in range(2):
            assert w.peval().VisitedSize == st.visited()
            np.testing.assert_array_equal(w.read(), st.val)
            np.testing.assert_array_equal(np.sign(w.flags()["active"]), np.sign(st.active))
    finally:
        w.close()
