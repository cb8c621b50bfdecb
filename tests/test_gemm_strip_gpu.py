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


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [(28_001, 113, 353), (64_530, 93, 99)])
def test_infinities_and_nan_stay_where_they_are(M, N, K, tb):
    """In op(B)'s first and last step and column, which the kernel reads again in place of what lies past them."""
    import torch
    from drone_amd import gcn
    gen = torch.Generator(device="cuda").manual_seed(K)
    A, B = torch.rand(M, K, generator=gen, device="cuda") + 0.5, torch.rand(K, N, generator=gen, device="cuda") + 0.5
    B[K - 1, 3], B[0, 5], B[K - 1, N - 1], B[7, N - 2] = float("inf"), float("nan"), float("-inf"), float("inf")
    got = gcn.sgemm(0, tb, A, B.t().contiguous() if tb else B)
    want = torch.full((N,), 1.0, device="cuda")
    want[3], want[5], want[N - 1], want[N - 2] = float("inf"), float("nan"), float("-inf"), float("inf")
    special = ~torch.isfinite(want)
    assert torch.isfinite(got[:, ~special]).all()
    for j in torch.nonzero(special).view(-1).tolist():
        assert torch.equal(torch.nan_to_num(got[:, j], nan=1.0, posinf=2.0, neginf=3.0), torch.nan_to_num(want[j], nan=1.0, posinf=2.0, neginf=3.0).expand(M))
