"""Chunks of short rows at the edges of what their bits hold: 1, 62, 63 and 64 rows, 15 ... 17 and 63 ... 65 entries together, rows without entries in
front, between, behind and alone, and rows of one entry to several batches, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lengths():
    one = [1] * 200
    rng = np.random.default_rng(5)
    yield "ones", one
    yield "empty", [0] * 130
    yield "gaps", ([0] + [1, 0, 0, 2] * 40 + [0] * 70 + [3] + [0] * 62 + [1] + [0] * 61 + [2] + [0] * 5)
    yield "edges", [63, 1, 64, 1, 0, 63, 0, 1, 65, 64, 0, 0, 16, 16, 16, 16, 15, 17, 32, 33, 1, 62, 1]
    yield "batches", [128, 129, 64, 192, 193, 1, 511, 512, 513, 0, 2, 1100, 0, 65, 66, 2300]
    yield "mixed", list(rng.choice([0, 0, 1, 1, 2, 3, 5, 9, 40, 64, 70], 3_000))


@pytest.mark.parametrize("name,lengths", list(_lengths()), ids=[n for n, _ in _lengths()])
def test_chunks(name, lengths):
    import torch
    from drone_amd import gcn
    rng = np.random.default_rng(len(lengths))
    n_cols = 3_000
    rp = np.zeros(len(lengths) + 1, np.int32)
    rp[1:] = np.cumsum(lengths)
    ci = rng.integers(0, n_cols, rp[-1]).astype(np.int32)
    val = rng.uniform(-1, 1, rp[-1]).astype(np.float32)
    dev = [torch.from_numpy(a).cuda() for a in (rp, ci, val)]
    row = np.repeat(np.arange(len(lengths)), lengths)
    for K in (1, 3, 4, 7, 16, 23, 40, 64, 100, 128, 200, 300):
        H = rng.uniform(-1, 1, (n_cols, K)).astype(np.float32)
        C0 = rng.uniform(-1, 1, (len(lengths), K + 3)).astype(np.float32)
        want, size = np.zeros((len(lengths), K)), np.zeros((len(lengths), K))
        np.add.at(want, row, val[:, None].astype(np.float64) * H[ci])
        np.add.at(size, row, np.abs(val[:, None].astype(np.float64) * H[ci]))
        plan = gcn.SpmmPlan(*dev, n_cols, K)
        for alpha, beta in ((1.0, 0.0), (0.75, -0.5)):
            out = torch.from_numpy(C0).cuda()
            gcn.spmm(plan, *dev, torch.from_numpy(H).cuda(), out=out[:, :K], alpha=alpha, beta=beta)
            got = out.cpu().numpy()
            # a row's sum takes at most its entries plus a dozen roundings of 2^-24 of the sum of its terms' sizes
            before = beta * C0[:, :K].astype(np.float64)
            bound = (np.asarray(lengths)[:, None] + 12) * 2.0 ** -24 * (abs(alpha) * size + np.abs(before))
            assert np.all(np.abs(got[:, :K] - (alpha * want + before)) <= bound), (K, beta)
            assert np.array_equal(got[:, K:], C0[:, K:]), (K, beta)
        plan.close()


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("rows", [4_500, 12_000, 24_000])
@pytest.mark.parametrize("longest", [339, 340, 512])
def test_longest_unsplit_row(longest, rows, split):
    """Either side of the line at which unsplit rows have more loads in flight, with and without split rows beside them, in lane groups of 8 to 32: a row's sum is
    taken in the same order either way, so the rows that two matrices share come out the same, bit by bit, and all of them right."""
    import scipy.sparse
    import torch
    from drone_amd import gcn
    rng = np.random.default_rng(rows)
    n_cols = 2_000
    lengths = rng.integers(0, 30, rows)
    lengths[::29] = rng.integers(65, 338, len(lengths[::29]))
    lengths[3], lengths[7], lengths[11] = 0, 64, 1_100 if split else 5
    at = lengths[:3].sum()
    ci, val = rng.integers(0, n_cols, lengths.sum()).astype(np.int32), rng.uniform(-1, 1, lengths.sum()).astype(np.float32)
    row_ci, row_val = rng.integers(0, n_cols, 512).astype(np.int32), rng.uniform(-1, 1, 512).astype(np.float32)
    for K in (23, 37, 64, 100, 128):
        H = rng.uniform(-1, 1, (n_cols, K)).astype(np.float32)
        got = []
        for lengths[3] in (longest, 338):
            rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
            c = np.insert(ci, at, row_ci[:lengths[3]])
            v = np.insert(val, at, row_val[:lengths[3]])
            dev = [torch.from_numpy(a).cuda() for a in (rp, c, v)]
            plan = gcn.SpmmPlan(*dev, n_cols, K)
            got.append(gcn.spmm(plan, *dev, torch.from_numpy(H).cuda()).cpu().numpy())
            plan.close()
            want = scipy.sparse.csr_matrix((v.astype(np.float64), c, rp), (rows, n_cols)) @ H.astype(np.float64)
            size = scipy.sparse.csr_matrix((np.abs(v).astype(np.float64), c, rp), (rows, n_cols)) @ np.abs(H).astype(np.float64)
            assert np.all(np.abs(got[-1] - want) <= (lengths[:, None] + 12) * 2.0 ** -24 * size), K  # as above
        others = np.arange(rows) != 3
        np.testing.assert_array_equal(got[0][others], got[1][others])


@pytest.mark.parametrize("longest", [3, 1_500])
def test_plan_is_whole_when_it_is_handed_out(longest):
    """Nothing of a plan is still being made on its stream when the call returns, with and without long rows: products may be on any other."""
    import torch
    from drone_amd import gcn
    n, K = 2_000_003, 8
    lengths = torch.arange(n, device="cuda", dtype=torch.int32) % 3
    lengths[n // 2] = longest
    rp = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    rp[1:] = torch.cumsum(lengths, 0)
    nnz = int(rp[-1])
    ci = (torch.arange(nnz, device="cuda") * 7919 % 1_000).to(torch.int32)
    val = (torch.arange(nnz, device="cuda") % 5 + 1).float()
    H = (torch.arange(1_000 * K, device="cuda").reshape(1_000, K) % 11).float()
    # whole numbers far below 2^24: exact in any order
    want = torch.zeros(n, K, device="cuda").index_add_(0, torch.repeat_interleave(torch.arange(n, device="cuda"), lengths), val[:, None] * H[ci.long()])
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(3):
        plan = gcn.SpmmPlan(rp, ci, val, 1_000, K, stream=side.cuda_stream)
        assert side.query()
        got = gcn.spmm(plan, rp, ci, val, H)
        assert torch.equal(got, want)
        plan.close()
