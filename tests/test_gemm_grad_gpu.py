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
    (128, 41, 60_001), (95, 5, 202_138), (1_000, 1_000, 700), (1_600, 1_280, 100), (2_000, 1_000, 70), (1_000, 2_200, 300)])
def test_blocks_splits_and_chains(M, N, K):
    _edges(1, 0, M, N, K)
