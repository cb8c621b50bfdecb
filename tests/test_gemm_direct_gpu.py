"""Products that sgemm_direct_kernel takes, at the edges of its tiles, pieces and reduction groups, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (transA, transB, M, N, K): every instance by rows / columns / reduction length, with one more and one less than whole
# blocks; K = 1 ... 17 and 15 mod 16 for the partial group, N = 33, 49, 97, 113 for pieces that slide back
CASES = ([(0, tb, m, n, k) for tb in (0, 1) for m, n, k in (
    (1, 1, 1), (16, 16, 16), (17, 15, 17), (100, 33, 31), (2708, 7, 64), (2708, 64, 1433), (515, 49, 400), (333, 80, 100),
    (1000, 97, 47), (300, 113, 383), (40_001, 17, 33), (30_011, 100, 65), (70_001, 61, 15), (20_000, 129, 385))] +
    [(1, 0, m, n, k) for m, n, k in (
        (2, 1, 5), (16, 16, 1000), (15, 7, 1281), (33, 16, 2708), (1433, 64, 2708), (65, 17, 3000), (47, 97, 5001),
        (320, 100, 30_011), (129, 65, 12_345), (31, 31, 70_001))])


@pytest.mark.parametrize("ta,tb,M,N,K", CASES)
def test_sgemm_direct_edges(ta, tb, M, N, K):
    import torch
    from drone_amd import gcn
    rng = np.random.default_rng(M * 131 + N * 7 + K)

    def padded(rows, cols, pad):  # row padding full of NaN: nothing may read it
        a = np.full((rows, cols + pad), np.nan, np.float32)
        a[:, :cols] = rng.standard_normal((rows, cols), dtype=np.float32)
        return torch.from_numpy(a).cuda(), a[:, :cols].astype(np.float64)

    A, a = padded(*((K, M) if ta else (M, K)), pad=M % 4)
    B, b = padded(*((N, K) if tb else (K, N)), pad=N % 3)
    a, b = a.T if ta else a, b.T if tb else b
    for alpha, beta, pad in ((1.0, 0.0, (16 - N) % 16), (0.75, -0.5, 3)):
        C0 = rng.standard_normal((M, N + pad), dtype=np.float32)
        C = torch.from_numpy(C0).cuda()
        again = C.clone()
        for out in (C, again):
            gcn.sgemm(ta, tb, A, B, out=out, alpha=alpha, beta=beta, M=M, N=N, K=K)
        got = C.cpu().numpy()
        want = alpha * (a @ b) + beta * C0[:, :N]
        # fp32 sums in any order: at most K + 2 roundings of 2^-24, each relative to the sum of magnitudes
        bound = (K + 2) * 2.0 ** -24 * (abs(alpha) * (np.abs(a) @ np.abs(b)) + abs(beta) * np.abs(C0[:, :N]))
        assert np.all(np.abs(got[:, :N] - want) <= bound)
        assert np.array_equal(got[:, N:], C0[:, N:]), "wrote into the padding"
        assert torch.equal(C, again)
