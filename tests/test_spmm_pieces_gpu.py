"""Long rows of the aggregation at the lengths where their pieces change: 512 entries (a row is cut at all), 128 and 256 (a
piece), 38,000 and 600,000 (a hub's pieces grow with it, up to 1,024), and 4,194,304 entries in long rows (column bands); and
short rows at the sizes of their chunks."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

SHORT = [512, 513, 639, 640, 641, 767, 769, 1024, 1025, 8191, 8193]
CASES = {
    "small": (SHORT + [1, 0, 64, 65], 20_011),
    "hub": (SHORT + [32_768, 33_000, 40_000, 300_000, 700_001], 700_001),
    "at_one_band": ([8192] * 512, 20_000),
    "bands": (SHORT + [8192] * 512, 70_001),
    # chunks of at most 16 entries, 16, 17 and 64 in a row; 32; no long row at all
    "chunks16": ([0, 1, 2, 13, 14, 15, 16, 17, 3, 0, 0, 63, 64, 65, 7, 9] * 9 + [600], 3001),
    "chunks32": ([0, 1, 15, 16, 17, 31, 32, 33, 2] * 1500 + [513, 700], 20_011),
    "no_long": ([1, 7, 16, 0, 40, 512] * 3, 1001),
    "bands_hub": ([8191] * 300 + [600, 513, 40_000, 300_000, 1_900_000], 1_900_003),
}


@pytest.mark.parametrize("K", [3, 41, 128])
@pytest.mark.parametrize("name", CASES)
def test_long_rows_at_their_edges(name, K):
    import torch
    from drone_amd import gcn
    lengths, n_cols = CASES[name]
    rng = np.random.default_rng(len(lengths) + K)
    lengths = rng.permutation(lengths)
    indptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    # distinct columns of a row: a random start and stride, coprime with n_cols; hot columns come first in every third row
    cols = []
    for i, d in enumerate(lengths):
        step = 1
        if i % 3:
            step = int(rng.integers(1, n_cols))
            while np.gcd(step, n_cols) != 1:
                step += 1
        cols.append(np.sort((int(rng.integers(n_cols)) * (i % 3) + np.arange(d, dtype=np.int64) * step) % n_cols))
    m = sp.csr_matrix((rng.uniform(-1, 1, indptr[-1]).astype(np.float32), np.concatenate(cols).astype(np.int32), indptr),
                      shape=(len(lengths), n_cols))
    B = rng.uniform(-1, 1, (n_cols, K)).astype(np.float32)
    C0 = rng.uniform(-1, 1, (len(lengths), K)).astype(np.float32)
    rp, ci, v, Bd, out = (torch.from_numpy(a).cuda() for a in (indptr, m.indices, m.data, B, C0.copy()))
    plan = gcn.SpmmPlan(rp, ci, v, n_cols, max_k=K)
    gcn.spmm(plan, rp, ci, v, Bd, K=K, out=out, alpha=1.5, beta=-0.5)
    again = torch.from_numpy(C0.copy()).cuda()
    gcn.spmm(plan, rp, ci, v, Bd, K=K, out=again, alpha=1.5, beta=-0.5)
    torch.cuda.synchronize()
    plan.close()
    assert torch.equal(out, again)  # sums have a fixed order
    m64, B64 = m.astype(np.float64), B.astype(np.float64)
    want = 1.5 * (m64 @ B64) - 0.5 * C0
    # a chain is at most 1,024 / 2 entries of a piece and 1,900 pieces: 2,400 roundings of 2^-24 each, 1.5e-4
    scale = 1.5 * (abs(m64) @ np.abs(B64)) + 0.5 * np.abs(C0)
    assert np.max(np.abs(out.cpu().numpy() - want) / np.maximum(scale, 1e-30)) <= 1.5e-4
