"""The one-launch-per-iteration layout of small fp64 PageRank plans, at the row lengths where its classes meet."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 7, 8, 9, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257, 1023, 1024, 1025, 1279, 1280, 1281]


@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("n,lengths,filler", [
    (6000, EDGES + [5000], 0),            # one row of every length at a class boundary, the rest empty: slices partly filled
    (6001, EDGES * 3, 3),                 # several of each among rows of 3
    (130_000, EDGES + [40_000, 511, 512, 513], 11),  # 1.5 M items: work-groups of 512
])
def test_pull_f64_row_length_classes(oracle, n, lengths, filler, deterministic):
    import torch
    from drone_amd.pagerank import PullPlanF64
    rng = np.random.default_rng(n)
    length = np.full(n, filler, np.int64)
    length[rng.choice(n, len(lengths), replace=False)] = lengths
    rp = np.zeros(n + 1, np.int64)
    rp[1:] = np.cumsum(length)
    ci = rng.integers(0, n - n // 5, rp[-1]).astype(np.int32)  # the last fifth dangles
    outdeg = np.bincount(ci, minlength=n)
    inv = np.where(outdeg > 0, 1.0 / np.maximum(outdeg, 1), 0.0)
    plan = PullPlanF64(torch.from_numpy(rp).cuda(), torch.from_numpy(ci).cuda(), torch.from_numpy(inv).cuda(),
                       deterministic=deterministic)
    for iters in (1, 2, 5):
        got = plan.run(0.85, iters).cpu().numpy()
        ref = oracle.pr_pull_f64(rp, ci, inv, 0.85, iters)
        # positive terms: a sum of L of them is within L * 2^-53 of exact in any order, twice that between two orders
        assert np.max(np.abs(got - ref) / ref) <= 2 * iters * max(length.max(), n // 256) * 2.0 ** -53
        assert np.array_equal(got, plan.run(0.85, iters).cpu().numpy())
    plan.close()
