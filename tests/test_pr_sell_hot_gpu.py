"""The fp64 PageRank iteration that keeps its hottest sources in LDS: more and fewer vertices than it keeps, odd counts, sources on
both sides of the last one kept, rows of every class and hub rows, and a matrix whose entries name too few of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEPT = 20_000
EDGES = [0, 1, 8, 9, 16, 17, 64, 65, 128, 129, 512, 513, 1023, 1024, 1025, 1279]


@pytest.mark.parametrize("n,filler,hot_share,more", [
    (15_001, 90, 1.0, [5000]),               # fewer than are kept
    (KEPT, 70, 1.0, [1025] * 300),           # as many; more hub rows than work-groups
    (KEPT + 1, 70, 1.0, []),
    (150_001, 9, 0.9, [40_000, 8193, 8192]),
    (150_002, 9, 0.62, [4097]),
    (150_003, 9, 0.2, [4097]),               # named too seldom: not kept
])
def test_hot_sources(oracle, n, filler, hot_share, more):
    import torch
    from drone_amd.pagerank import PullPlanF64
    rng = np.random.default_rng(n)
    length = np.full(n, filler, np.int64)
    first = rng.permutation(n)[:KEPT + 500]  # the rows of most entries: they are numbered first
    length[first] += 1 + np.arange(len(first))[::-1] % 3
    length[rng.choice(n, len(EDGES + more), replace=False)] = EDGES + more
    rp = np.zeros(n + 1, np.int64)
    rp[1:] = np.cumsum(length)
    by_length = np.argsort(-length, kind="stable")
    m = int(rp[-1])
    assert n + m > 1200 << 10
    rank = np.where(rng.random(m) < hot_share, rng.integers(0, min(KEPT, n), m), rng.integers(min(KEPT, n - 1), n - (n > KEPT + 1) * (n // 5), m))
    rank[:2000] = np.clip(KEPT - 3 + np.arange(2000) % 6, 0, n - 1)  # on both sides of the last one kept
    ci = by_length[rank].astype(np.int32)
    outdeg = np.bincount(ci, minlength=n)
    inv = np.where(outdeg > 0, 1.0 / np.maximum(outdeg, 1), 0.0)
    plan = PullPlanF64(torch.from_numpy(rp).cuda(), torch.from_numpy(ci).cuda(), torch.from_numpy(inv).cuda())
    for iters in (1, 2, 5):
        got = plan.run(0.85, iters).cpu().numpy()
        ref = oracle.pr_pull_f64(rp, ci, inv, 0.85, iters)
        # positive terms: a sum of L of them is within L * 2^-53 of exact in any order, twice that between two orders
        assert np.max(np.abs(got - ref) / ref) <= 2 * iters * max(length.max(), n // 256) * 2.0 ** -53
        assert np.array_equal(got, plan.run(0.85, iters).cpu().numpy())
    plan.close()


@pytest.mark.parametrize("n,more", [(9_001, []), (9_002, [4095, 4096, 4097, 8999]), (700, [699])])
def test_hub_rows_of_small_matrices(oracle, n, more):
    """Rows around the length from which a work-group takes them, and around one and two rounds of its gathers."""
    import torch
    from drone_amd.pagerank import PullPlanF64
    rng = np.random.default_rng(n)
    length = rng.integers(0, 12, n)
    at = [767, 768, 769] * (n > 1000) + more
    length[rng.choice(n, len(at), replace=False)] = at
    rp = np.concatenate([[0], np.cumsum(length)]).astype(np.int64)
    ci = np.concatenate([rng.permutation(n)[:d] for d in length]).astype(np.int32)
    outdeg = np.bincount(ci, minlength=n)
    inv = np.where(outdeg > 0, 1.0 / np.maximum(outdeg, 1), 0.0)
    plan = PullPlanF64(torch.from_numpy(rp).cuda(), torch.from_numpy(ci).cuda(), torch.from_numpy(inv).cuda())
    for iters in (1, 2, 5):
        got = plan.run(0.85, iters).cpu().numpy()
        ref = oracle.pr_pull_f64(rp, ci, inv, 0.85, iters)
        # as above
        assert np.max(np.abs(got - ref) / ref) <= 2 * iters * max(length.max(), 64) * 2.0 ** -53
    plan.close()
