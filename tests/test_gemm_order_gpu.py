"""The order in which the products that share a result with another kernel add up: sgemm_strip_kernel, sgemm_flat_kernel and sgemm_twin_kernel take the
steps of a reduction as the kernels do that they stand in for, so that a product has the same bits on either side of a rule's line.  Against chains of
fused multiply-adds on the host, and against the other kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _groups(first, end, K):
    """Steps of groups of 16: for j = 0 ... 3 the quarters in turn (sgemm_direct_kernel)."""
    return [k for g in range(first, end) for j in range(4) for k in range(16 * g + j, 16 * g + 16, 4) if k < K]


def _order(order, K):
    """The chains of steps whose sums are added one after the other."""
    if order == "ascending":  # sgemm_mfma_kernel
        return [list(range(K))]
    if order == "groups":
        return [_groups(0, (K + 15) // 16, K)]
    whole = K // 16
    chains = [_groups(whole * s // 8, whole * (s + 1) // 8, K) for s in range(8)]
    chains[-1] += _groups(whole, whole + 1, K)
    return chains


def _chain(a, b, steps):
    """Fused multiply-adds: a product of floats is exact in 64 bits of mantissa, and so is, but for 1 in 2^40, what decides the one rounding."""
    acc = np.zeros(len(a), np.float32)
    for k in steps:
        acc = (a[:, k].astype(np.longdouble) * b[:, k] + acc).astype(np.float32)
    return acc


def _operands(tb, M, N, K):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(M + 131 * N + K)
    return torch.randn(M, K, generator=gen, device="cuda"), torch.randn(*((N, K) if tb else (K, N)), generator=gen, device="cuda")


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K,order", [
    # flat: instead of the tiled kernel, of the direct one; groups in part, reductions of 1 ... 3 steps
    (24_000, 50, 13, "ascending"), (30_011, 41, 16, "ascending"), (40_000, 100, 23, "ascending"), (24_000, 128, 3, "ascending"),
    (8_000, 116, 7, "groups"), (28_000, 13, 50, "groups"), (24_000, 40, 38, "groups"), (24_001, 13, 64, "groups"),
    # strip
    (30_011, 100, 320, "ascending"), (40_000, 62, 576, "ascending"), (30_000, 128, 301, "ascending"),
    (28_200, 32, 224, "groups"), (64_530, 93, 99, "groups"), (100_000, 23, 92, "groups"),
    # twin: every width, shares of unlike length, a group in part
    (1_726, 16, 1_440, "shares"), (1_726, 25, 1_441, "shares"), (4_090, 48, 400, "shares"), (3_986, 68, 1_104, "shares"), (4_090, 96, 415, "shares"),
    (2_748, 117, 1_452, "shares"), (376, 112, 1_201, "shares"), (2_708, 64, 1_440, "shares")])
def test_steps_are_added_in_order(tb, M, N, K, order):
    from drone_amd import gcn
    A, B = _operands(tb, M, N, K)
    got = gcn.sgemm(0, tb, A, B).cpu().numpy()
    rng = np.random.default_rng(K)
    i = np.concatenate([[0, 0, M - 1, M - 1], rng.integers(0, M, 28), np.full(16, M - 1)])
    j = np.concatenate([[0, N - 1, 0, N - 1], rng.integers(0, N, 28), np.maximum(N - 1 - np.arange(16), 0)])  # with the pieces that slide back
    a, b = A.cpu().numpy()[i], (B if tb else B.t()).cpu().numpy()[j]
    want = np.zeros(len(i), np.float32)
    for steps in _order(order, K):
        want = want + _chain(a, b, steps)
    np.testing.assert_array_equal(got[i, j], want)


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [(24_000, 50, 13), (40_000, 100, 23), (8_000, 116, 7), (28_000, 13, 50), (24_003, 49, 33), (45_001, 82, 48), (28_001, 63, 64)])
def test_flat_gives_the_bits_of_a_product_with_beta(tb, M, N, K):
    """Which the other kernels take."""
    import torch
    from drone_amd import gcn
    A, B = _operands(tb, M, N, K)
    zeros = torch.zeros(M, N, device="cuda")
    assert torch.equal(gcn.sgemm(0, tb, A, B), gcn.sgemm(0, tb, A, B, out=zeros, beta=1.0))


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K,fewer", [(28_000, 128, 320, 27_999), (28_000, 100, 300, 27_999), (28_015, 113, 353, 27_990),  # strip / tiled
                                         (28_200, 32, 224, 27_990),                                                           # strip / direct
                                         (4_097, 16, 400, 4_096), (4_200, 80, 527, 4_096), (5_000, 96, 640, 2_048)])          # direct / twin
def test_rows_have_the_same_bits_on_either_side_of_a_line(tb, M, N, K, fewer):
    import torch
    from drone_amd import gcn
    A, B = _operands(tb, M, N, K)
    assert torch.equal(gcn.sgemm(0, tb, A, B)[:fewer], gcn.sgemm(0, tb, A[:fewer], B))
