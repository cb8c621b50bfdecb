"""Forward products at the lines of sgemm_strip_kernel's rule and blocks: its fewest rows, strips of 16 rows and columns with one more or
less, reductions of one group of 16 up to pieces that slide back by 1 ... 15 steps, op(B) that just fits the LDS and that does not, B
in both layouts, and sums in the order of either kernel that it stands in for."""
import pytest

from test_gemm_direct_gpu import test_sgemm_direct_edges as _edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [
    (28_000, 94, 31), (28_001, 128, 320), (27_999, 128, 320), (28_015, 113, 353), (43_777, 128, 16), (60_000, 97, 17), (90_001, 81, 18), (55_333, 65, 79),
    (120_001, 49, 45), (90_001, 33, 62), (140_003, 17, 36), (140_000, 16, 36), (70_001, 1, 1_150), (65_537, 96, 426), (40_001, 112, 365),
    (33_333, 64, 640), (33_333, 64, 641)])
def test_strips_and_pieces(tb, M, N, K):
    _edges(0, tb, M, N, K)
