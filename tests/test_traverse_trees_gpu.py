"""CC_PEVal where labels come from joining trees: graphs whose edges all have their reverse, with rows on both sides of every
length at which they are dealt out differently, long chains, many components, and graphs in which one edge has no reverse.
Labels are whole numbers: exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _both(u, v):
    return np.concatenate([u, v]), np.concatenate([v, u])


def _named(u, v, seed):
    """Random names, edges in random order."""
    rng = np.random.default_rng(seed)
    perm, order = rng.permutation(int(max(u.max(), v.max())) + 1), rng.permutation(len(u))
    return perm[u][order].astype(np.int32), perm[v][order].astype(np.int32)


def _grid(w, h):
    at = np.arange(w * h).reshape(h, w)
    return _both(np.concatenate([at[:-1].ravel(), at[:, :-1].ravel()]), np.concatenate([at[1:].ravel(), at[:, 1:].ravel()]))


def _path(n):
    return _both(np.arange(n - 1), np.arange(1, n))


def _stars(degrees):
    """Stars of the given numbers of leaves, the centres chained through their last leaves."""
    u, v, at = [], [], 0
    for d in degrees:
        u += [at] * d
        v += range(at + 1, at + d + 1)
        if at + d + 1 < sum(degrees) + len(degrees):
            u.append(at + d)
            v.append(at + d + 1)
        at += d + 1
    return _both(np.array(u), np.array(v))


def _blocks(sizes, seed):
    """Components of the given sizes: a random tree and as many edges more, some of them twice and from a vertex to itself."""
    rng = np.random.default_rng(seed)
    u, v, base = [], [], 0
    for k in sizes:
        child = np.arange(1, k)
        more = rng.integers(0, k, (2, k))
        u += [base + child, base + more[0], base + more[0][:3]]
        v += [base + (rng.random(k - 1) * child).astype(np.int64), base + more[1], base + more[1][:3]]
        base += k
    return _both(np.concatenate(u), np.concatenate(v))


CASES = {
    "pair": lambda: _both(np.array([0]), np.array([1])),
    "samples": lambda: _path(65),
    "path_in_order": lambda: tuple(x.astype(np.int32) for x in _path(70_001)),
    "path": lambda: _named(*_path(30_011), 1),
    "grid": lambda: _named(*_grid(211, 97), 2),
    "rows": lambda: _named(*_stars([1, 7, 8, 9, 63, 64, 65, 255, 257, 511, 2047, 2048, 2049, 9000]), 3),
    "components": lambda: _named(*_blocks([2] * 300 + [3, 17, 1000, 40_000] * 3, 4), 5),
    "one_by_one": lambda: _named(*_blocks([2] * 40_000, 6), 7),
    # falling and rising turns: roots that are joined to one another in a long row
    "comb": lambda: _both(np.concatenate([np.arange(0, 20_000), np.arange(1, 20_000)]),
                          np.concatenate([40_000 + np.arange(0, 20_000), 40_000 + np.arange(0, 19_999)])),
}


def _labels(n, index, dst):
    src = np.repeat(np.arange(n), np.diff(index))
    cc = np.arange(n)
    while True:  # least label over in-edges, and the label of that label
        new = cc.copy()
        np.minimum.at(new, dst, cc[src])
        new = np.minimum(new, new[new])
        if np.array_equal(new, cc):
            return cc
        cc = new


@pytest.mark.parametrize("without_reverse", [0, 1, 2])
@pytest.mark.parametrize("name", CASES)
def test_labels_by_trees(oracle, name, without_reverse):
    from drone_amd.traverse import CCWorkerCUDA
    u, v = (np.asarray(x, np.int32) for x in CASES[name]())
    if without_reverse == 1:  # one edge leads one way
        u, v = u[:-1], v[:-1]
    elif without_reverse == 2:  # many do
        keep = np.random.default_rng(8).random(len(u)) < 0.9
        keep[0] = True
        u, v = u[keep], v[keep]
    nglobal = int(max(u.max(), v.max())) + 1
    n, _, _, index, dst = oracle.build_graph(nglobal, u, v)
    want = _labels(n, index, dst)
    w = CCWorkerCUDA(nglobal, u, v)
    try:
        for _ in range(3):
            res = w.peval()
            np.testing.assert_array_equal(w.read(), want)
            flags = w.flags()
            np.testing.assert_array_equal(flags["active"] > 0, want < np.arange(n))
            assert not flags["updateByMessage"].any()
            assert res.VisitedSize == np.count_nonzero(want < np.arange(n))
    finally:
        w.close()


@pytest.mark.parametrize("other_is_hub", [False, True])
@pytest.mark.parametrize("into_the_largest", [True, False])
@pytest.mark.parametrize("size", [10, 100, 3_000])
def test_one_edge_without_reverse_between_components(oracle, size, into_the_largest, other_is_hub):
    """A component of most vertices and a small one, joined by one edge that leads one way and is not the least of its row."""
    from drone_amd.traverse import CCWorkerCUDA
    rng = np.random.default_rng(size)
    small, large = np.arange(0, size, dtype=np.int32), np.arange(size, 40 * size, dtype=np.int32)
    if not into_the_largest:  # the one way leads from smaller to larger labels
        small, large = np.arange(39 * size, 40 * size, dtype=np.int32), np.arange(0, 39 * size, dtype=np.int32)

    def connected(names, hub):  # a star, or a random tree
        k = np.arange(1, len(names))
        up = np.zeros(len(k), np.int64) if hub else (rng.random(len(k)) * k).astype(np.int64)
        return _both(names[k], names[up])

    # local numbers go by first appearance
    us, vs = zip(*sorted([connected(small, other_is_hub), connected(large, False)], key=lambda e: e[0].min()))
    one = (small[-1], large[-1]) if into_the_largest else (large[-1], small[-1])
    u, v = np.concatenate([*us, [one[0]]]).astype(np.int32), np.concatenate([*vs, [one[1]]]).astype(np.int32)
    n, l2g, _, index, dst = oracle.build_graph(40 * size, u, v)
    want = _labels(n, index, dst)
    assert want.max() == 0  # the edge joins them, though one way only
    w = CCWorkerCUDA(40 * size, u, v)
    try:
        for _ in range(2):
            w.peval()
            np.testing.assert_array_equal(w.read(), want)
    finally:
        w.close()


@pytest.mark.parametrize("one_way", [0.0, 0.02, 0.3])
@pytest.mark.parametrize("first_tree", ["few", "half", "most"])
def test_edges_of_the_first_tree_need_not_lead_back(oracle, first_tree, one_way):
    """Random graphs whose vertex 0 is in the tree of few, half or most of the vertices, by edges of which some lead one way, and
    whose other edges have their reverse, all but some: what the tree of vertex 0 is made of is not looked up in the other direction."""
    from drone_amd.traverse import CCWorkerCUDA
    rng = np.random.default_rng([len(first_tree), int(100 * one_way)])
    for n in (2, 3, 65, 700, 5_000, 70_003):
        first = rng.permutation(np.arange(1, n))[:int(n * {"few": 0.05, "half": 0.5, "most": 0.95}[first_tree])]
        down_u, down_v = np.zeros(len(first), np.int64), first           # 0 -> its tree
        back = rng.random(len(first)) >= max(one_way, 0.3)               # some of them lead back
        a, b = rng.integers(0, n, (2, n // 3 + 1))                       # any two vertices, this edge
        there = rng.random(len(a)) >= one_way                            # and its reverse
        own = np.arange(n)                                               # (numbers go by first appearance)
        u = np.concatenate([own, down_u, down_v[back], a, b[there]]).astype(np.int32)
        v = np.concatenate([own, down_v, down_u[back], b, a[there]]).astype(np.int32)
        _, l2g, _, index, dst = oracle.build_graph(n, u, v)
        assert np.array_equal(l2g, own)
        want = _labels(n, index, dst)
        w = CCWorkerCUDA(n, u, v)
        try:
            for _ in range(2):
                w.peval()
                np.testing.assert_array_equal(w.read(), want)
                np.testing.assert_array_equal(w.flags()["active"] > 0, want < own)
        finally:
            w.close()


def test_one_way_edge_into_a_root_that_is_joined_before_its_row_is_due(oracle):
    """Rows come to cc_link's work-groups 64 at a time, piece i to work-group i mod 2,048, and past 524,288 vertices a work-group has a second
    round of them.  Here work-group 0 has a row of half a million entries in its first round and vertex r in its second; by then
    work-group 1 has looked at the vertex that an edge leads from to r, one way, and, in its second round, joined r to the tree that most
    samples lie in, whose vertices are left out.  The edge carries the least label into all of that tree."""
    from drone_amd.traverse import CCWorkerCUDA
    work_groups, piece, samples = 2048, 64, 64
    second = 4 * work_groups * piece
    n = second + 16 * piece
    largest, hub, r, y, q, z = 2, 3, second, second + piece, second + piece + 1, second + 5 * piece
    own = np.arange(n)
    sampled = own[::n // samples][1:samples]
    sampled = sampled[sampled < second]
    many = np.setdiff1d(np.arange(2 * piece, second), sampled)
    pairs = [(0, q), (r, y), (y, z), (largest, z)] + [(largest, int(v)) for v in sampled]
    a, b = np.concatenate([np.array(pairs).T, np.stack([np.full_like(many, hub), many])], 1)
    u, v = np.concatenate([own, a, b, [q]]).astype(np.int32), np.concatenate([own, b, a, [r]]).astype(np.int32)
    _, l2g, _, index, dst = oracle.build_graph(n, u, v)
    assert np.array_equal(l2g, own)
    want = _labels(n, index, dst)
    assert want[r] == want[y] == want[z] == want[largest] == 0 and np.all(want[sampled] == 0) and np.all(want[many] == hub)
    for _ in range(3):  # (a graph that has shown an edge without its reverse is not tried again)
        w = CCWorkerCUDA(n, u, v)
        try:
            w.peval()
            np.testing.assert_array_equal(w.read(), want)
        finally:
            w.close()
