"""A product with a scaled plan (band pieces, short-row chunks, bit core on the plan's side stream) recorded into a HIP
graph and replayed: every replay must give the bits of the eager call."""
import numpy as np
import pytest

from test_gcn_gpu import _core_graph, dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import torch
    return torch


def test_spmm_with_bit_core_in_a_hip_graph(T):
    from drone_amd import gcn
    rng = np.random.default_rng(5)
    n, K = 12000, 128
    rp, cols, in_deg, out_deg = _core_graph(rng, n, 6000, 0.8, 60000)
    d_rp, d_ci = dev(T, rp), dev(T, cols)
    d_val = gcn.edge_values(d_rp, d_ci, dev(T, in_deg), dev(T, out_deg))
    plan = gcn.SpmmPlan(d_rp, d_ci, d_val, n, max_k=K, row_scale=gcn.degree_scales(dev(T, out_deg)),
                        col_scale=gcn.degree_scales(dev(T, in_deg)))
    assert plan.bit_core()["cells"] > 0
    B = T.rand((n, K), device="cuda") * 2 - 1
    eager = gcn.spmm(plan, d_rp, d_ci, d_val, B)
    T.cuda.synchronize()
    out = T.zeros((n, K), device="cuda")
    side = T.cuda.Stream()
    graph = T.cuda.CUDAGraph()
    with T.cuda.stream(side):
        gcn.spmm(plan, d_rp, d_ci, d_val, B, out=out, stream=side.cuda_stream)   # warm-up on the capture stream
        side.synchronize()
        with T.cuda.graph(graph, stream=side):
            gcn.spmm(plan, d_rp, d_ci, d_val, B, out=out, stream=side.cuda_stream)
    for it in range(4):
        out.fill_(float(it))                          # the program's own eager work between the replays
        T.cuda.synchronize()
        graph.replay()
        T.cuda.synchronize()
        assert T.equal(out, eager), it
        B2 = B * (1.0 + it)                           # new operand values through the same buffer
        want = gcn.spmm(plan, d_rp, d_ci, d_val, B2)
        T.cuda.synchronize()
        B.copy_(B2)
        graph.replay()
        T.cuda.synchronize()
        assert T.equal(out, want), it
        eager = want
    plan.close()


@pytest.mark.parametrize("deterministic", [False, True])
def test_pagerank_iterations_in_a_hip_graph(T, deterministic):
    """Twenty iterations of the fp64 pull PageRank (sweep, merge of shared blocks, fix-up with the last work-group's
    reduction) recorded once and replayed: the deterministic mode bit for bit, the default mode to 1e-12 per vertex
    (its LDS additions are not ordered)."""
    from drone_amd import rmat
    from drone_amd.pagerank import PullPlanF64
    x = rmat.pagerank_inputs_torch(14, 16, 3)
    side = T.cuda.Stream()
    T.cuda.synchronize()
    plan = PullPlanF64(x["row_ptr"], x["col_idx"], x["inv_outdeg"], deterministic=deterministic, shared_blocks=True)
    eager = plan.run(0.85, 20)
    T.cuda.synchronize()
    out = T.zeros_like(eager)
    plan.stream = side.cuda_stream
    graph = T.cuda.CUDAGraph()
    with T.cuda.stream(side):
        plan.run(0.85, 20, out=out)
        side.synchronize()
        with T.cuda.graph(graph, stream=side):
            plan.run(0.85, 20, out=out)
    for it in range(3):
        out.zero_()
        T.cuda.synchronize()
        graph.replay()
        T.cuda.synchronize()
        if deterministic:
            assert T.equal(out, eager), it
        else:
            assert float(((out - eager).abs() / eager).max()) <= 1e-12, it
    plan.close()


def test_first_loss_on_a_stream_is_recorded(T):
    """The first loss of a stream is recorded, not run: the scratch it makes has to be ready for the calls that are run before
    (and between) the replays."""
    from drone_amd._lib import check, lib
    n, classes = 5000, 7
    gen = T.Generator(device="cuda").manual_seed(3)
    z = T.randn(n, classes, generator=gen, device="cuda")
    truth = T.randint(0, classes, (n,), generator=gen, device="cuda", dtype=T.int32)
    want = float(T.nn.functional.cross_entropy(z.double(), truth.long()))
    loss, count = T.zeros(1, device="cuda"), T.zeros(1, dtype=T.int32, device="cuda")
    junk = T.full((1 << 20,), -1, dtype=T.int32, device="cuda")
    T.cuda.synchronize()
    del junk
    T.cuda.empty_cache()
    side, graph = T.cuda.Stream(), T.cuda.CUDAGraph()

    def call():
        check(lib().drone_cross_entropy_f32(n, classes, z.data_ptr(), classes, truth.data_ptr(), None, classes, 1.0, loss.data_ptr(),
                                            count.data_ptr(), side.cuda_stream))

    def result():
        T.cuda.synchronize()
        got = float(loss), int(count)
        loss.zero_(), count.zero_()
        T.cuda.synchronize()
        assert got[1] == n and abs(got[0] - want) <= 1e-6 * want  # fp32 exp and log of values near 1, summed in fp64

    with T.cuda.graph(graph, stream=side, capture_error_mode="relaxed"):
        call()
    for _ in range(3):
        call()
        result()
        graph.replay()
        result()


@pytest.mark.parametrize("M,N,K", [(1_317, 194, 1_792), (128, 41, 60_001)])
def test_first_split_product_on_a_stream_is_recorded(T, M, N, K):
    """The first product of a stream whose reduction is split is recorded: its scratch is allocated under the capture, and stays where it is when a larger product
    asks for more."""
    from drone_amd import gcn
    gen = T.Generator(device="cuda").manual_seed(M)
    A, B = T.randn(K, M, generator=gen, device="cuda"), T.randn(K, N, generator=gen, device="cuda")
    A2, B2 = T.randn(30_011, 640, generator=gen, device="cuda"), T.randn(30_011, 200, generator=gen, device="cuda")
    A3, B3 = T.cat([A2, A2], 1), T.cat([B2, B2], 1)
    want, want2, want3 = (gcn.sgemm(True, False, *ab) for ab in ((A, B), (A2, B2), (A3, B3)))
    out, out2 = T.zeros(M, N, device="cuda"), T.zeros(640, 200, device="cuda")
    out3 = T.zeros(1_280, 400, device="cuda")
    T.cuda.synchronize()
    side, graph, second = T.cuda.Stream(), T.cuda.CUDAGraph(), T.cuda.CUDAGraph()
    with T.cuda.graph(graph, stream=side):
        gcn.sgemm(True, False, A, B, out=out, stream=side.cuda_stream)
    with T.cuda.graph(second, stream=side):
        gcn.sgemm(True, False, A2, B2, out=out2, stream=side.cuda_stream)
    with T.cuda.stream(side):  # all of it in order
        for _ in range(3):
            graph.replay()
            side.synchronize()
            assert T.equal(out, want)
            out.zero_()
            second.replay()
            gcn.sgemm(True, False, A, B, out=out, stream=side.cuda_stream)
            side.synchronize()
            assert T.equal(out2, want2) and T.equal(out, want)
            out.zero_(), out2.zero_()
            gcn.sgemm(True, False, A3, B3, out=out3, stream=side.cuda_stream)
            side.synchronize()
            assert T.equal(out3, want3)
