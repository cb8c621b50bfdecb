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
