"""Rounds of CC_PEVal and SSSP_PEVal at the list and row sizes where the kernel that runs them changes: a lone wavefront up to
64 edges, one work-group up to 4,096, then the whole GPU, then sweeps; in a sweep over the open vertices rows up to 8, 256 and
4,096 entries and longer ones.  Labels and distances are whole numbers below 2^24: exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _layers(widths, fan, seed):
    """Vertices in layers of the given widths; every vertex of a layer is entered from up to `fan` of the layer before."""
    rng = np.random.default_rng(seed)
    u, v, base = [], [], 0
    for a, b in zip(widths[:-1], widths[1:]):
        k = min(fan, a)
        src = base + (np.arange(b)[:, None] * k + np.arange(k)[None, :]) % a
        u.append(src.ravel())
        v.append(np.repeat(base + a + np.arange(b), k))
        base += a
    u, v = np.concatenate(u), np.concatenate(v)
    perm = rng.permutation(base + widths[-1])  # labels do not follow the layers
    perm[[0, np.flatnonzero(perm == 0)[0]]] = perm[[np.flatnonzero(perm == 0)[0], 0]]
    return perm[u].astype(np.int32), perm[v].astype(np.int32)


def _rows(lengths, sources):
    """A start vertex, `sources` vertices it reaches, then rows of the given in-degrees fed by them, by vertices that nothing
    reaches, or by both with the reached one at either end."""
    u, v = [np.zeros(sources, np.int64)], [np.arange(1, sources + 1)]
    dead, at = 1 + sources + 4 * len(lengths), 1 + sources
    for d in lengths:
        for how in range(4):
            src = dead + np.arange(d)
            if how == 0:
                src = 1 + np.arange(d)
            elif how == 1:
                src[0] = 1 + d % sources
            elif how == 2:
                src = np.sort(np.append(dead + np.arange(d - 1), 1 + d % sources)) if d > 1 else np.array([1])
            u.append(src)
            v.append(np.full(len(src), at))
            at += 1
    u, v = np.concatenate(u), np.concatenate(v)
    n = dead + max(lengths)
    perm = np.random.default_rng(len(u)).permutation(n)  # the reached in-neighbour may stand anywhere in its row
    return perm[u].astype(np.int32), perm[v].astype(np.int32)


CASES = {
    "lone": lambda: _layers([1] + [63, 64, 65] * 3, 1, 1),
    # few edges per vertex on average, many per vertex, for the lone wavefront; lists that leave it and come back
    "chain": lambda: _layers([1] * 40 + [2, 5, 1, 9, 13, 1, 64, 1, 65, 1, 4, 16, 16, 3] * 3, 4, 6),
    "chain_many": lambda: _layers([1] * 40 + [2, 5, 1, 9, 13, 1, 64, 1, 65, 1, 4, 16, 16, 3] * 3 + [300, 3000, 3000], 12, 7),
    # labels that come from as far as a first round looks, from one hop further and from much further away
    "falling": lambda: (np.concatenate([np.arange(31), 100 + np.arange(32), 200 + np.arange(33), 300 + np.arange(500), [0, 0, 0]]).astype(np.int32),
                        np.concatenate([np.arange(1, 32), 101 + np.arange(32), 201 + np.arange(33), 301 + np.arange(500), [100, 200, 300]]).astype(np.int32)),
    "group": lambda: _layers([1, 31, 65, 255, 1024, 1025, 2048, 64, 1365, 1366, 1, 1], 3, 2),
    "edge4096": lambda: _layers([1, 4096, 4096, 4097, 4097, 2, 4096, 4095], 1, 3),
    "device": lambda: _layers([1, 3000, 9000, 9001, 9000, 300, 70_000, 69_999, 40, 1], 2, 4),
    "wide": lambda: _layers([1, 200_000, 600_001, 1_000_000, 300_000, 20], 1, 5),
    "rows": lambda: _rows([1, 7, 8, 9, 15, 16, 17, 32, 33, 255, 256, 257, 4095, 4096, 4097, 8193], 20_000),
}


def _bellman(index, dst, start, length):
    src = np.repeat(np.arange(len(index) - 1), np.diff(index))
    dist = np.full(len(index) - 1, 1e8, np.float32)
    dist[start] = 0
    while True:
        new = dist.copy()
        np.minimum.at(new, dst, dist[src] + length)
        if np.array_equal(new, dist):
            return dist
        dist = new


@pytest.mark.parametrize("name", CASES)
def test_rounds_at_their_edges(oracle, name):
    from drone_amd.traverse import CCWorkerCUDA, SSSPWorkerCUDA
    u, v = CASES[name]()
    nglobal, start = int(max(u.max(), v.max())) + 1, int(u[0])
    n, g2l, l2g, index, dst = oracle.build_graph(nglobal, u, v)
    ones = np.ones(len(dst), np.float32)
    whole = np.random.default_rng(9).integers(1, 5, len(dst)).astype(np.float32)
    w = SSSPWorkerCUDA(nglobal, u, v, startId=start)
    try:
        for length in (ones, whole):
            w.set_edge_len(length)
            want = _bellman(index, dst, int(g2l[start]), length)
            for _ in range(2):  # the state of a call must not outlive it
                res = w.peval()
                np.testing.assert_array_equal(w.read(), want)
                assert res.VisitedSize == n - 1  # all but the start vertex, whose flag stays 0
    finally:
        w.close()
    cc = np.arange(n)
    src = np.repeat(np.arange(n), np.diff(index))
    while True:
        new = cc.copy()
        np.minimum.at(new, dst, cc[src])
        if np.array_equal(new, cc):
            break
        cc = new
    w = CCWorkerCUDA(nglobal, u, v)
    try:
        for _ in range(2):
            res = w.peval()
            np.testing.assert_array_equal(w.read(), cc)
            assert res.VisitedSize == np.count_nonzero(cc != np.arange(n))
    finally:
        w.close()


def _near_ties(copies, filler):
    """A start vertex and `copies` of x -> y -> z, where x falls in the first round and once more in the third: by less than
    the tolerance of 1e-6, by more, or by both along two edges.  Edges with lengths; filler: as many edges that nothing reaches."""
    e = []
    for i in range(copies):
        a, b, c, d, x, y, z = range(1 + 7 * i, 8 + 7 * i)
        e += [(0, a, 1.0), (a, c, 0.5), (c, x, 0.5), (x, y, 1.0), (y, z, 1.0)]
        e.append((0, x, [2 + 2 ** -21, 2 + 2 ** -18, 2 + 2 ** -18][i % 3]))  # c brings 2.0: 4.8e-7, 3.8e-6 below
        if i % 3 == 2:
            e += [(0, b, 1.0), (b, d, 0.5), (d, x, 0.5 + 2 ** -18 - 2 ** -21)]  # 4.8e-7 below
    base = 1 + 7 * copies
    at = np.arange(filler)
    u, v, w = (np.array(c) for c in zip(*e))
    u = np.concatenate([u, base + at % 1000])
    v = np.concatenate([v, base + 1000 + at // 1000])
    w = np.concatenate([w, np.ones(filler)]).astype(np.float32)
    perm = np.random.default_rng(copies).permutation(int(max(u.max(), v.max())) + 1)
    return perm[u].astype(np.int32), perm[v].astype(np.int32), w


@pytest.mark.parametrize("kind,copies,filler", [("lone", 3, 0), ("lone", 13, 0), ("group", 40, 0), ("group", 1200, 0),
                                                ("device", 3000, 200_000), ("sweep", 6000, 0)])
def test_improvements_within_the_tolerance(oracle, kind, copies, filler):
    """Every kind of listed round stores an improvement of at most 1e-6 and does not carry it on, as sssp.cu:62-68: the same
    distances and flags as the oracle's, whichever kernel runs the round.  A sweep takes it along."""
    from drone_amd.traverse import SSSPWorkerCUDA
    u, v, length = _near_ties(copies, filler)
    nglobal, start = int(max(u.max(), v.max())) + 1, int(u[0])
    n, g2l, l2g, index, dst = oracle.build_graph(nglobal, u, v)
    by_edge = {(a, b): w for a, b, w in zip(u.tolist(), v.tolist(), length.tolist())}
    src = np.repeat(np.arange(n), np.diff(index))
    local = np.array([by_edge[e] for e in zip(l2g[src].tolist(), l2g[dst].tolist())], np.float32)
    st = oracle.SSSPState(index, dst, local)
    st.peval(int(g2l[start]))
    exact = _bellman(index, dst, int(g2l[start]), local)
    assert (exact < st.val).sum() == 2 * ((copies + 2) // 3)  # y and z of the copies that fall by little
    w = SSSPWorkerCUDA(nglobal, u, v, startId=start)
    try:
        w.set_edge_len(local)
        for _ in range(2):
            res = w.peval()
            got = w.read()
            if kind == "sweep":
                assert (exact <= got).all() and (got <= st.val).all()
            else:
                np.testing.assert_array_equal(got, st.val)
                np.testing.assert_array_equal(np.sign(w.flags()["active"]), np.sign(st.active))
            assert res.VisitedSize == st.visited()
    finally:
        w.close()


def test_cycle_that_falls_within_the_tolerance():
    """A cycle whose length is negative by less than the tolerance ends after one turn, without an error (sssp.cu:64)."""
    from drone_amd import _lib
    from drone_amd.traverse import SSSPWorkerCUDA
    w = SSSPWorkerCUDA(3, np.array([0, 1, 2], np.int32), np.array([1, 2, 0], np.int32), startId=0)
    try:
        w.set_edge_len(np.array([1.0, 1.0, -2 - 2 ** -21], np.float32))
        w.peval()
        assert _lib.lib().drone_last_error() == 0
        np.testing.assert_array_equal(w.read(), np.array([-2 ** -21, 1.0, 2.0], np.float32))
    finally:
        w.close()


@pytest.mark.parametrize("pairs,more", [((8 << 20) // 2, 32), ((8 << 20) // 2 + 1, 0)])
def test_memory_of_large_graphs_is_bounded(pairs, more):
    """What the first call keeps per vertex: its state (three words), four words of lists and, up to 8 Mi vertices, 32 bytes of
    first edges.  Pairs of vertices, one edge each."""
    import torch
    from drone_amd.traverse import CCWorkerCUDA
    u = np.arange(0, 2 * pairs, 2, dtype=np.int32)
    w = CCWorkerCUDA(2 * pairs, u, u + 1)
    try:
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        res = w.peval()
        kept = before - torch.cuda.mem_get_info()[0]
        want = 2 * pairs * (12 + 16 + more)
        assert abs(kept - want) <= 24 << 20, (kept, want)  # allocations come in pieces of at least 2 MB
        assert res.VisitedSize == pairs
        np.testing.assert_array_equal(w.read(), np.arange(2 * pairs) // 2 * 2)
    finally:
        w.close()
