"""Row synchronisation in place (workers of one loopback group): row widths around the lane groups, padded rows, the most
workers it takes and one more, and tables that do not agree with each other, against the oracle bit for bit."""
import numpy as np
import pytest

from partition_util import vertex_cut

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("compress", [False, True])
@pytest.mark.parametrize("W,Ks,agree", [(2, (1, 15, 16, 17), True), (3, (31, 32, 33, 7), True), (16, (63, 64, 65, 130), True),
                                        (17, (5, 33), True), (4, (9, 40), False)])
def test_rows_direct(oracle, W, Ks, agree, compress):
    import torch
    from drone_amd import gcn, rmat
    from drone_amd._lib import lib
    from drone_amd.pagerank import Loopback, run_workers
    from drone_amd.traverse import _WorkerCUDA
    n = 1 << 9
    u, v = rmat.clean_directed_np(*rmat.rmat_edges(9, 8 << 9, seed=W))
    parts, _ = vertex_cut(u, v, W, W)
    parts = [{k: np.array(a) for k, a in p.items()} for p in parts]
    if not agree:  # a master forgets one of its mirrors: the mirror's row is still added, but not written back
        # (on the worker with the most mirrors of its own: it has staging for one more row than its lists name)
        p = max(parts, key=lambda q: len(q["mirror_vertex"]) - len(q["mirror_workers"]))
        assert len(p["mirror_vertex"]) > len(p["mirror_workers"])
        at = int(np.argmax(p["mirror_number"]))
        assert p["mirror_number"][at] >= 2
        p["mirror_workers"] = np.delete(p["mirror_workers"], int(p["mirror_number"][:at].sum()))
        p["mirror_number"][at] -= 1
    tops = [oracle.Part(oracle.build_graph(n, p["u"], p["v"])[2], n, p["master_vertex"], p["mirror_number"], p["mirror_workers"],
                        p["mirror_vertex"], p["master_worker"]) for p in parts]
    sizes = [len(oracle.build_graph(n, p["u"], p["v"])[2]) for p in parts]
    rng = np.random.default_rng(W)
    lb = Loopback(W, timeout_ms=60000)
    ws = [_WorkerCUDA(n, p["u"], p["v"], workerId=i, workerNum=W, routes=p, loopback=lb) for i, p in enumerate(parts)]
    try:
        for K in Ks:
            host = [rng.standard_normal((nl, K)).astype(np.float32) for nl in sizes]
            full = [torch.full((nl, K + i % 3), 7.0, device="cuda") for i, nl in enumerate(sizes)]
            for f, h in zip(full, host):
                f[:, :K] = torch.from_numpy(h)
            torch.cuda.synchronize()
            want = oracle.graphsum_sync_rows(tops, host, compress=compress)
            got = run_workers([(lambda i=i: gcn.graphsum_sync_rows(ws[i].g, full[i][:, :K], i, W, ws[i].comm, compress))
                               for i in range(W)])
            for i in range(W):
                assert got[i] == (want[0][i], want[1][i])
                np.testing.assert_array_equal(full[i][:, :K].cpu().numpy(), host[i])
                assert (full[i][:, K:] == 7.0).all()
    finally:
        for w in ws:
            lib().drone_graph_destroy(w.g)
            w.g = None
        lb.close()


@pytest.mark.parametrize("compress", [False, True])
def test_chains_of_masters_take_the_general_path(oracle, compress):
    """Tables that agree item by item, but where a worker's master is itself a mirror of another's (C's mirror names A, A's own
    row is a mirror of B's): two workers would write A's row at once, so nothing is summed in place."""
    import torch
    from drone_amd import gcn, rmat
    from drone_amd._lib import lib
    from drone_amd.pagerank import Loopback, run_workers
    from drone_amd.traverse import _WorkerCUDA
    n, W, K = 1 << 9, 3, 37
    u, v = rmat.clean_directed_np(*rmat.rmat_edges(9, 8 << 9, seed=5))
    parts, master = vertex_cut(u, v, W, 5)
    lists = [({int(x): [] for x in p["master_vertex"]}, dict(zip(p["mirror_vertex"].tolist(), p["master_worker"].tolist()))) for p in parts]
    for w, (_, mirrors) in enumerate(lists):
        for x, b in mirrors.items():
            lists[b][0][x].append(w)
    chained = 0
    for x, b in master.items():
        if len(lists[b][0].get(x, [])) == 2:
            a, c = lists[b][0][x]
            lists[b][0][x], lists[a][0][x], lists[c][1][x] = [a], [c], a
            chained += 1
    assert chained > 50
    for p, (masters, mirrors) in zip(parts, lists):
        p.update(master_vertex=np.array(sorted(masters), np.int32), mirror_number=np.array([len(masters[x]) for x in sorted(masters)], np.int32),
                 mirror_workers=np.array([w for x in sorted(masters) for w in masters[x]], np.int32),
                 mirror_vertex=np.array(sorted(mirrors), np.int32), master_worker=np.array([mirrors[x] for x in sorted(mirrors)], np.int32))
    local = [oracle.build_graph(n, p["u"], p["v"])[2] for p in parts]
    tops = [oracle.Part(l2g, n, p["master_vertex"], p["mirror_number"], p["mirror_workers"], p["mirror_vertex"], p["master_worker"])
            for l2g, p in zip(local, parts)]
    rng = np.random.default_rng(7)
    lb = Loopback(W, timeout_ms=60000)
    ws = [_WorkerCUDA(n, p["u"], p["v"], workerId=i, workerNum=W, routes=p, loopback=lb) for i, p in enumerate(parts)]
    try:
        host = [rng.standard_normal((len(l2g), K)).astype(np.float32) for l2g in local]
        rows = [torch.from_numpy(h.copy()).cuda() for h in host]
        torch.cuda.synchronize()
        want = oracle.graphsum_sync_rows(tops, host, compress=compress)
        got = run_workers([(lambda i=i: gcn.graphsum_sync_rows(ws[i].g, rows[i], i, W, ws[i].comm, compress)) for i in range(W)])
        for i in range(W):
            assert got[i] == (want[0][i], want[1][i])
            np.testing.assert_array_equal(rows[i].cpu().numpy(), host[i])
    finally:
        for w in ws:
            lib().drone_graph_destroy(w.g)
            w.g = None
        lb.close()


def test_workers_that_disagree_about_the_rows_get_an_error():
    """Different widths, or compressed rows on one side only: every worker gets an error instead of waiting, and the group goes on
    working."""
    import torch
    from drone_amd import gcn, rmat
    from drone_amd._lib import DroneError, lib
    from drone_amd.pagerank import Loopback, run_workers
    from drone_amd.traverse import _WorkerCUDA
    n, W = 1 << 9, 3
    u, v = rmat.clean_directed_np(*rmat.rmat_edges(9, 8 << 9, seed=5))
    parts, _ = vertex_cut(u, v, W, 5)
    lb = Loopback(W, timeout_ms=20000)
    ws = [_WorkerCUDA(n, p["u"], p["v"], workerId=i, workerNum=W, routes=p, loopback=lb) for i, p in enumerate(parts)]
    try:
        rows = [torch.ones(w.n, 8, device="cuda") for w in ws]
        torch.cuda.synchronize()

        def sync(i, K, compress):
            try:
                return gcn.graphsum_sync_rows(ws[i].g, rows[i][:, :K], i, W, ws[i].comm, compress)
            except DroneError as e:
                return str(e)

        for K, compress in (((8, 8, 7), (False,) * 3), ((8, 8, 8), (False, True, False))):
            got = run_workers([(lambda i=i: sync(i, K[i], compress[i])) for i in range(W)])
            assert all(isinstance(g, str) and "different exchange steps" in g for g in got)
            assert all(bool((r == 1.0).all()) for r in rows)
        got = run_workers([(lambda i=i: sync(i, 8, False)) for i in range(W)])
        assert [g[1] for g in got] == [len(p["mirror_vertex"]) for p in parts]
    finally:
        for w in ws:
            lib().drone_graph_destroy(w.g)
            w.g = None
        lb.close()
