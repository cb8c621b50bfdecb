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
