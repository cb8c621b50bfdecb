"""Deep products of few rows at the lines of sgemm_twin_kernel's rule and blocks: every width by rows and columns, with one more and one less than
whole tiles and than 256 blocks, shares of unlike length, reductions that end in a group of 1 ... 15 steps, B in both layouts; and shorter
reductions whose blocks are halved to fill the CUs."""
import pytest

from test_gemm_direct_gpu import test_sgemm_direct_edges as _edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [
    (1, 1, 384), (16, 16, 399), (17, 128, 400), (4_096, 16, 385), (4_097, 16, 400), (2_048, 32, 511), (2_049, 33, 496), (1_365, 48, 415),
    (1_361, 49, 1_433), (3_985, 65, 512), (4_090, 80, 527), (2_033, 97, 640), (2_049, 96, 641), (4_095, 127, 768), (4_096, 128, 1_000),
    (255, 113, 383), (1_884, 25, 137), (2_040, 17, 64)])
def test_twin_shares_and_widths(tb, M, N, K):
    _edges(0, tb, M, N, K)
