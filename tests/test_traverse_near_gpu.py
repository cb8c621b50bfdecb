"""Distances over natural lengths by rounds of the nearest vertices first (NearRounds), where its lists, thresholds and waiting vertices are at their
limits: grids, a vertex with more edges than a list may have, one with just as many, more waiting vertices than there is room for, lists that are cut,
lengths of zero and near 2^24 (distances that round and that pass the unreached one), and lengths below zero, which take the other rounds.
They begin after 64 rounds.  Against the oracle, exactly: sums of whole numbers in float have one least fixed point, in whatever order they are made."""
import numpy as np
import pytest

from test_traverse_rounds_gpu import _layers

pytestmark = pytest.mark.gpu


def _grid(w, h):
    at = np.arange(w * h).reshape(h, w)
    s = np.concatenate([at[:-1].ravel(), at[:, :-1].ravel()])
    d = np.concatenate([at[1:].ravel(), at[:, 1:].ravel()])
    return np.concatenate([s, d]).astype(np.int32), np.concatenate([d, s]).astype(np.int32)


def _hub(before, edges, tail):
    """A path to a vertex with `edges` out-edges, each leading to a path of `tail` vertices."""
    ends = before + 1 + np.arange(edges)[:, None] + edges * np.arange(tail)[None, :]
    u = np.concatenate([np.arange(before), np.full(edges, before), ends[:, :-1].ravel()])
    v = np.concatenate([np.arange(1, before + 1), ends[:, 0], ends[:, 1:].ravel()])
    return u.astype(np.int32), v.astype(np.int32)


def _detour(edges, tail):
    """A path to a fan of 100; one of the fan leads to a path of `tail` vertices by a long edge, and by two short ones through a vertex with `edges` out-edges, which finds no room on a list beside the path's first."""
    fan, hub, leaf = 64 + np.arange(100), 164, 165 + np.arange(edges - 1)
    path = 165 + edges - 1 + np.arange(tail + 1)
    u = np.concatenate([np.arange(63), np.full(100, 63), [64], fan, [hub], np.full(edges - 1, hub), path[:-1]])
    v = np.concatenate([np.arange(1, 64), fan, [path[0]], np.where(fan == 64, hub, 0), [path[0]], leaf, path[1:]])
    return u.astype(np.int32), v.astype(np.int32)


def _detour_lengths(n, g2l, l2g, index, dst):
    length = np.ones(len(dst), np.float32)
    at = lambda u, v: [e for e in range(index[g2l[u]], index[g2l[u] + 1]) if l2g[dst[e]] == v]
    head = max(l2g[dst[e]] for e in range(index[g2l[64]], index[g2l[64] + 1]))
    length[at(64, head)] = 100.0
    length[at(63, 65)] = 1 << 20  # the first threshold lies beyond the path
    return length


@pytest.mark.parametrize("edges", [2048, 2100])
def test_long_path_lowered_twice(oracle, edges):
    """More rounds than there are vertices, some by the nearest vertices first and some not: no cycle of negative length."""
    from drone_amd.traverse import SSSPWorkerCUDA
    u, v = _detour(edges, 5000)
    nglobal = int(max(u.max(), v.max())) + 1
    n, g2l, l2g, index, dst = oracle.build_graph(nglobal, u, v)
    length = _detour_lengths(n, g2l, l2g, index, dst)
    st = oracle.SSSPState(index, dst, length)
    st.peval(int(g2l[0]))
    assert st.val[g2l[nglobal - 1]] == 63 + 1 + 1 + 1 + 5000
    w = SSSPWorkerCUDA(nglobal, u, v, startId=0)
    try:
        w.set_edge_len(length)
        assert w.peval().VisitedSize == st.visited()
        np.testing.assert_array_equal(w.read(), st.val)
    finally:
        w.close()


def test_list_cut_before_its_first_entry(oracle):
    """A vertex with more edges than a list may have, lowered alone while another waits, leaves a list of none.  The rounds of the nearest go on with the other one's path, a round a
    hop, and the large vertex comes last, by the other rounds: a list that still counted it would have no room for the path, and the large vertex's turn would come first."""
    from drone_amd.traverse import SSSPWorkerCUDA
    fan, way, tail, leaves = 64 + np.arange(100), 164 + np.arange(6), 170 + np.arange(500), 670 + np.arange(2_100)
    hub, far = way[-1], fan[-1]
    u = np.concatenate([np.arange(63), np.full(100, 63), fan, way[:-1], np.full(2_100, hub), tail[:-1]]).astype(np.int32)
    v = np.concatenate([np.arange(1, 64), fan, [way[0]], np.zeros(98), [tail[0]], way[1:], leaves, tail[1:]]).astype(np.int32)
    nglobal = 670 + 2_100
    n, g2l, l2g, index, dst = oracle.build_graph(nglobal, u, v)
    length = np.ones(len(dst), np.float32)
    length[[e for e in range(index[g2l[63]], index[g2l[63] + 1]) if l2g[dst[e]] == far]] = 1 << 20  # waits while the others are done
    length[index[g2l[0]]] = 2.0  # (not all are 1)
    st = oracle.SSSPState(index, dst, length)
    st.peval(int(g2l[0]))
    w = SSSPWorkerCUDA(nglobal, u, v, startId=0)
    try:
        w.set_edge_len(length)
        for _ in range(2):
            w.peval()
            np.testing.assert_array_equal(w.read(), st.val)
            round_of = w.flags()["active"]
            assert round_of[g2l[leaves]].min() > round_of[g2l[tail[-1]]]
    finally:
        w.close()


CASES = {
    "grid_3": (lambda: _grid(3, 300), 1, 17), "grid_23": (lambda: _grid(23, 211), 1, 17), "grid_120": (lambda: _grid(120, 130), 1, 17),
    "grid_600": (lambda: _grid(600, 60), 1, 17),           # lists that are cut
    "ones_and_two": (lambda: _grid(40, 50), 1, 3), "zeros": (lambda: _grid(31, 57), 0, 4), "far": (lambda: _grid(17, 40), 1, 1 << 24),
    "hub_2048": (lambda: _hub(99, 2048, 3), 1, 5), "hub_2049": (lambda: _hub(99, 2049, 3), 1, 5), "hub_late": (lambda: _hub(700, 3000, 2), 1, 5),
    "waiting": (lambda: _layers([1] * 70 + [500, 2047, 4000, 4100, 300, 2], 1, 3), 1, 400), "waiting_more": (lambda: _layers([1] * 70 + [60, 1900, 3900, 3900, 40], 2, 8), 1, 60),
    "places": (lambda: _layers([1] * 70 + [40, 900, 1000, 1000, 900, 900] + [30, 900, 1000, 600] * 3, 3, 9), 1, 17),  # more entries than vertices, but for the sifting
    "negative": (lambda: _layers([1] * 70 + [30, 300, 300, 50, 2], 2, 4), -3, 9), "path": (lambda: (np.arange(3000, dtype=np.int32), np.arange(1, 3001, dtype=np.int32)), 1, 9),
}


@pytest.mark.parametrize("name", CASES)
def test_nearest_first(oracle, name):
    from drone_amd.traverse import SSSPWorkerCUDA
    make, low, high = CASES[name]
    u, v = make()
    nglobal = int(max(u.max(), v.max())) + 1
    n, g2l, l2g, index, dst = oracle.build_graph(nglobal, u, v)
    length = np.random.default_rng(len(u)).integers(low, high, len(dst)).astype(np.float32)
    if name == "waiting":
        length[::7] = 1.0
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
