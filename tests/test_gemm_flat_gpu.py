"""Short rows on both sides at the lines of sgemm_flat_kernel's rule and blocks: its fewest rows instead of the tiled and instead of the direct kernel,
every number of groups and tiles, last pieces of columns that slide back, reductions of 1 ... 3 steps and pieces that slide back by 1 ... 15, a last
strip of one row, B in both layouts, and (with a beta, as every second product of a case has) what the other kernels do with them."""
import pytest

from test_gemm_direct_gpu import test_sgemm_direct_edges as _edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [
    (8_000, 128, 1), (8_001, 113, 2), (7_999, 97, 3), (9_999, 65, 4), (12_001, 81, 5), (24_000, 50, 13), (23_999, 7, 31), (24_001, 1, 17), (30_011, 100, 23),
    (40_017, 17, 15), (33_333, 33, 16), (33_333, 16, 32), (70_001, 64, 29), (24_003, 49, 33), (50_002, 31, 47), (45_001, 82, 48), (60_001, 96, 46),
    (45_001, 34, 62), (28_001, 63, 64), (100_001, 2, 63), (60_507, 81, 62)])
def test_strips_pieces_and_groups(tb, M, N, K):
    _edges(0, tb, M, N, K)
