"""Weight gradients at the lines where sgemm_grad_kernel's blocks, splits and chains of additions change: single rows and columns, blocks
that reach past the output, (split, block) counts that the eight XCDs do not divide, groups of 16 rows short of one for every
wavefront, and one more or less than the groups of a chain or a round."""
import pytest

from test_gemm_direct_gpu import test_sgemm_direct_edges as _edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (1, 1, 1), (1, 1, 5_000), (1, 130, 300), (130, 1, 17), (3, 2, 100_000), (16, 16, 15), (16, 17, 16), (17, 16, 17), (17, 17, 63),
    (17, 33, 64), (33, 17, 65), (33, 33, 255), (32, 64, 256), (31, 63, 257), (65, 33, 511), (97, 41, 512), (129, 17, 513),
    (60, 48, 4 * 12 * 16), (60, 48, 4 * 13 * 16 - 1), (60, 48, 4 * 13 * 16), (640, 94, 8_000), (333, 100, 4 * 13 * 16 * 12), (333, 100, 4 * 14 * 16 * 12 + 5),
    (128, 41, 60_001), (95, 5, 202_138), (1_000, 1_000, 700), (1_600, 1_280, 100), (2_000, 1_000, 70), (1_000, 2_200, 300),
    # blocks of 32 tiles: 24, 25, 26, 48, 49 and 50 groups a wavefront, whose chains have 24
    (616, 396, 10_673), (633, 388, 11_338), (1_291, 400, 4_970), (1_259, 394, 9_198), (1_280, 397, 9_434), (1_277, 386, 9_596)])
def test_blocks_splits_and_chains(M, N, K):
    _edges(1, 0, M, N, K)


@pytest.mark.parametrize("M,N,K", [(900, 450, 20_011), (1_358, 235, 73_123), (602, 128, 232_965)])
def test_no_chain_of_additions_is_long(M, N, K):
    """Products of 1 + 2^-14, whose sums are exact in float up to 512 of them and lose 2^-14 with each from 1,024 on.  A wavefront's chains of additions have at
    most 384 rows, so what is lost is a rounding of 2^-24 for each chain, wavefront and split that joins a sum; chains of all the rows of a split's
    quarter lost 1e-5 to 5e-5 of it."""
    import torch
    from drone_amd import gcn
    a, b = torch.pow(2.0, torch.arange(M) % 5 - 2), (1 + 2.0 ** -14) * (1 - 2 * (torch.arange(N) % 2))
    A, B = a.cuda().expand(K, M).contiguous(), b.cuda().expand(K, N).contiguous()
    want = K * torch.outer(a.double(), b.double())
    got = gcn.sgemm(True, False, A, B).cpu().double()
    joins = K / 384 / 4 + 1 + 4 + 32  # of all chains of a wavefront if there were one split, and up to 32 splits
    assert float(((got - want) / want).abs().max()) <= joins * 2.0 ** -24
