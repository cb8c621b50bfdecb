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
