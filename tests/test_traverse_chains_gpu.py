"""SSSP_PEVal over unit lengths where most vertices lie in chains, which are taken in one step: chains that end in one vertex
twice, side by side, in rings without an end, entered from the middle, one-way or doubled in places, and the same graphs with
other lengths.  Distances are whole numbers below 2^24: exact."""
import heapq

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dijkstra(n, index, dst, length, start):
    dist, heap = [1e8] * n, [(0.0, start)]
    dist[start] = 0.0
    while heap:
        d, v = heapq.heappop(heap)
        if d > dist[v]:
            continue
        for e in range(index[v], index[v + 1]):
            if d + length[e] < dist[dst[e]]:
                dist[dst[e]] = d + length[e]
                heapq.heappush(heap, (dist[dst[e]], dst[e]))
    return np.array(dist, np.float32)


class _Roads:
    def __init__(self):
        self.edges, self.n = [], 0

    def crossing(self):
        self.n += 1
        return self.n - 1

    def road(self, a, b, inner):
        """A chain of `inner` vertices from a to b, every edge in both directions; returns them."""
        on = list(range(self.n, self.n + inner))
        self.n += inner
        way = [a] + on + [b]
        for x, y in zip(way[:-1], way[1:]):
            self.edges += [(x, y), (y, x)]
        return on

    def ring(self, size):
        on = list(range(self.n, self.n + size))
        self.n += size
        for x, y in zip(on, on[1:] + on[:1]):
            self.edges += [(x, y), (y, x)]
        return on


def _path(n, at):
    r = _Roads()
    a, b = r.crossing(), r.crossing()
    on = r.road(a, b, n - 2)
    return r, ([a] + on + [b])[at]


def _mixed(start):
    r = _Roads()
    c = [r.crossing() for _ in range(6)]
    ways = [r.road(c[0], c[1], 40), r.road(c[0], c[1], 41), r.road(c[1], c[2], 300), r.road(c[2], c[2], 77), r.road(c[2], c[3], 1),
            r.road(c[3], c[3], 2), r.road(c[3], c[4], 500), r.road(c[4], c[0], 260), r.road(c[0], c[0], 3)]
    ring, small = r.ring(300), r.ring(3)
    one_way = r.road(c[4], c[5], 90)
    r.edges.remove((one_way[50], one_way[51]))  # only the way back
    doubled = r.road(c[5], c[1], 90)
    r.edges += [(doubled[10], doubled[11])]
    entered = r.road(c[5], c[4], 60)
    r.edges += [(c[0], entered[30]), (entered[40], c[3])]
    r.edges += [(ways[2][9], ways[2][9])]  # to itself
    return r, dict(crossing=c[2], middle=ways[6][123], beside=ways[0][3], loop=ways[3][70], alone=ways[4][0], ring=ring[7], small=small[0],
                   dead_end=one_way[70], last=ways[7][-1])[start]


def _star(arms, inner):
    r = _Roads()
    centre = r.crossing()
    for k in range(arms):
        r.road(centre, r.crossing(), inner + k % 5)
    return r, 1 + centre


CASES = {**{f"path{n}_{at}": (lambda n=n, at=at: _path(n, at)) for n, at in ((256, 0), (257, 100), (5000, 4999), (20_011, 7777))},
         **{f"mixed_{s}": (lambda s=s: _mixed(s)) for s in ("crossing", "middle", "beside", "loop", "alone", "ring", "small", "dead_end", "last")},
         "star": lambda: _star(300, 17), "star_many": lambda: _star(5000, 9)}


@pytest.mark.parametrize("name", CASES)
def test_distances_over_chains(oracle, name):
    from drone_amd.traverse import SSSPWorkerCUDA
    roads, start = CASES[name]()
    rng = np.random.default_rng(len(roads.edges))
    perm, order = rng.permutation(roads.n), rng.permutation(len(roads.edges))
    edges = perm[np.array(roads.edges)][order].astype(np.int32)
    u, v = np.ascontiguousarray(edges[:, 0]), np.ascontiguousarray(edges[:, 1])
    start = int(perm[start])
    n, g2l, l2g, index, dst = oracle.build_graph(roads.n, u, v)
    ones, whole = np.ones(len(dst), np.float32), rng.integers(1, 9, len(dst)).astype(np.float32)
    w = SSSPWorkerCUDA(roads.n, u, v, startId=start)
    try:
        for length in (ones, ones, whole, whole, ones):
            w.set_edge_len(length)
            want = _dijkstra(n, index, dst, length, int(g2l[start]))
            res = w.peval()
            np.testing.assert_array_equal(w.read(), want)
            flags = w.flags()["active"]
            assert flags[g2l[start]] == 0
            np.testing.assert_array_equal(flags > 0, (want < 1e8) & (np.arange(n) != g2l[start]))
            assert res.VisitedSize == n - 1
    finally:
        w.close()
