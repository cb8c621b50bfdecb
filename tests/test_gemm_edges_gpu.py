"""Tiles that reach past the matrix: the last row and column tiles of the tiled GEMM at every remainder of a 16-byte piece,
whole and partial last steps of the reduction, in all four orientations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(n, n, k) for n in (1, 2, 3, 4, 5, 63, 65, 126, 127, 129, 130, 131, 132, 133) for k in (64, 96, 97)]
                         + [(40_001, 100, 320), (40_002, 101, 301), (40_003, 126, 320), (33_001, 131, 224), (131, 133, 20_000)])
@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_edge_tiles(tA, tB, M, N, K):
    import torch
    from drone_amd import gcn
    rng = np.random.default_rng(M + N + K)
    A, B = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    C0 = rng.uniform(-1, 1, (M, N + 3)).astype(np.float32)
    # poison around the operands: nothing of it may reach an output
    def held(a):
        big = torch.full((a.shape[0] + 1, a.shape[1] + 3), float("nan"), device="cuda")
        big[:a.shape[0], :a.shape[1]] = torch.from_numpy(np.ascontiguousarray(a)).cuda()
        return big[:a.shape[0], :a.shape[1]]
    dA, dB = held(A.T if tA else A), held(B.T if tB else B)
    out = torch.from_numpy(C0.copy()).cuda()
    gcn.sgemm(tA, tB, dA, dB, out=out[:, :N], alpha=0.75, beta=-0.5)
    got = out.cpu().numpy()
    want = 0.75 * (A.astype(np.float64) @ B) - 0.5 * C0[:, :N]
    # K + 2 roundings of 2^-24 of the sum of the products' sizes
    bound = (K + 2) * 2.0 ** -24 * (0.75 * (np.abs(A).astype(np.float64) @ np.abs(B)) + 0.5 * np.abs(C0[:, :N]))
    assert np.all(np.abs(got[:, :N] - want) <= bound)
    assert np.array_equal(got[:, N:], C0[:, N:])
