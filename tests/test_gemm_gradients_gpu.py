"""Weight gradients (A transposed) from single blocks to many and over short and long reductions, with outputs and reductions of one more or less than
whole tiles and groups of 16; and forward products in 64-row tiles and over deep reductions."""
import pytest

from test_gemm_direct_gpu import test_sgemm_direct_edges as _edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (64, 30, 255), (64, 17, 256), (65, 32, 127), (65, 31, 129), (65, 32, 4097),
    (32, 33, 2000), (33, 64, 2001), (63, 64, 128), (64, 64, 36_621), (64, 64, 36_622), (64, 63, 36_000),
    (32, 128, 122_071), (33, 128, 118_372), (301, 127, 13_080), (301, 127, 13_079), (317, 115, 13_717), (67, 65, 9_001), (61, 96, 9_000),
    (1400, 100, 3_572), (1400, 128, 127), (16, 16, 257), (17, 16, 255)])
def test_weight_gradients(M, N, K):
    _edges(1, 0, M, N, K)


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [(49_152, 128, 300), (49_153, 127, 300), (24_513, 129, 65), (4_097, 900, 97), (65, 3_001, 1_001), (63, 3_001, 1_000),
                                   (12_345, 70, 1_100), (700, 40, 1_471), (700, 57, 384 + 16 * 8 + 5)])
def test_rows_of_half_tiles_and_deep_reductions(M, N, K, tb):
    _edges(0, tb, M, N, K)
