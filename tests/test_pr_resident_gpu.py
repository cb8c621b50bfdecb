"""Runs of small fp64 PageRank plans, whose work-groups stay for the whole run: at the edges of what a lane stages, with more slices
and hub rows than work-groups, recorded into a graph, and by the work-groups that came before the gate was closed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(n, lengths, filler):
    """Row lengths `lengths` at random places among rows of `filler` entries; the last fifth of the vertices dangles."""
    rng = np.random.default_rng(n + filler)
    length = np.full(n, filler, np.int64)
    length[rng.choice(n, len(lengths), replace=False)] = lengths
    rp = np.zeros(n + 1, np.int64)
    rp[1:] = np.cumsum(length)
    ci = rng.integers(0, max(1, n - n // 5), rp[-1]).astype(np.int32)
    outdeg = np.bincount(ci, minlength=n)
    return rp, ci, np.where(outdeg > 0, 1.0 / np.maximum(outdeg, 1), 0.0)


def _plan(rp, ci, inv):
    import torch
    from drone_amd.pagerank import PullPlanF64
    return PullPlanF64(torch.from_numpy(rp).cuda(), torch.from_numpy(ci).cuda(), torch.from_numpy(inv).cuda())


def _close(got, ref, rp, iters):
    # positive terms: a sum of L of them is within L * 2^-53 of exact in any order, twice that between two orders
    n = len(ref)
    assert np.max(np.abs(got - ref) / ref) <= 2 * iters * max(np.diff(rp).max(), n) * 2.0 ** -53


@pytest.mark.parametrize("n,lengths,filler", [
    (1, [], 0), (1, [], 3), (2, [1], 0), (65, [64, 768, 769], 2),
    (1023, [2048, 2049, 1, 0], 5), (1024, [], 0), (1025, [12, 13, 96], 9),
    (4096, [800] * 64, 3), (4097, [800] * 65, 11),           # as many hub rows as work-groups, and one more
    (6000, [30_000, 5000, 4096, 4097], 1),                   # hub rows of several rounds
    (8192, [], 60), (8200, [], 60),                          # as many slices as wavefronts, and one more
    (12288, [768] * 5, 11), (12289, [768] * 5, 11),          # as many rows as fit
    (19455, [9] * 1024, 0), (14000, [12] * 6000, 0),         # most rows without entries: too many of them to fit, and not
    (1000, [], 768), (1650, [], 768), (1400, [], 900),       # slices as long as the kernel keeps, and matrices that have longer ones
])
def test_runs_in_one_launch(oracle, n, lengths, filler):
    rp, ci, inv = _matrix(n, lengths, filler)
    plan = _plan(rp, ci, inv)
    for iters in (1, 2, 3, 4, 5, 8, 9, 10):
        got = plan.run(0.85, iters).cpu().numpy()
        _close(got, oracle.pr_pull_f64(rp, ci, inv, 0.85, iters), rp, iters)
        assert np.array_equal(got, plan.run(0.85, iters).cpu().numpy())
    plan.close()


@pytest.mark.parametrize("n,lengths,filler", [(700, [900, 2100], 4), (6000, [800] * 64, 12), (8192, [], 60)])
def test_as_many_work_groups_as_found_a_place(oracle, n, lengths, filler):
    from drone_amd._lib import check, lib
    rp, ci, inv = _matrix(n, lengths, filler)
    plan = _plan(rp, ci, inv)
    for iters in (1, 2, 5, 6):
        got = []
        # runs behind a gate closed at so many, or at whoever has come by the first look, and open ones follow each other
        for patience, places in ((64, 1), (64, 1000), (64, 2), (0, 1000), (64, 3), (64, 63), (0, 64), (64, 1000)):
            check(lib().drone_pr_plan_gate(plan.h, patience, places))
            got.append(plan.run(0.85, iters).cpu().numpy())
            _close(got[-1], oracle.pr_pull_f64(rp, ci, inv, 0.85, iters), rp, iters)
            assert np.array_equal(got[0], got[-1])
    plan.close()


@pytest.mark.parametrize("iters", [3, 4, 5, 6, 9])
def test_a_wait_in_vain_is_reported_and_leaves_the_plan_clean(iters):
    """Work-groups that wait for nothing: the next run says so, and those after it find no value of that run."""
    import torch
    from drone_amd._lib import check, lib
    plan = _plan(*_matrix(6000, [800] * 64, 12))
    want = plan.run(0.85, iters)
    for _ in range(3):
        check(lib().drone_pr_plan_gate(plan.h, -1, 64))  # the 64 of its hub rows
        plan.run(0.85, iters)
        torch.cuda.synchronize()
        with pytest.raises(RuntimeError, match="waited in vain"):
            plan.run(0.85, iters)
        check(lib().drone_pr_plan_gate(plan.h, 64, 64))
        for _ in range(3):
            assert torch.equal(plan.run(0.85, iters), want)
    plan.close()


def test_a_busy_chip_costs_places_and_not_the_run():
    """Beside a stream that keeps every CU busy some work-groups are late, and the others do not leave the run to one of them: it takes
    less than a third of what it takes one (0.3 of 8.6 ms where measured)."""
    import time
    import torch
    from drone_amd._lib import check, lib
    plan = _plan(*_matrix(12000, [], 28))
    main, other = torch.cuda.Stream(), torch.cuda.Stream()
    plan.stream = main.cuda_stream
    out, big = torch.empty(12000, dtype=torch.float64, device="cuda"), torch.zeros(1 << 28, device="cuda")
    median = {}
    for places in (1, 64):
        check(lib().drone_pr_plan_gate(plan.h, 64, places))
        plan.run(0.85, 20, out=out)
        times = []
        while len(times) < 9:
            torch.cuda.synchronize()
            with torch.cuda.stream(other):
                for _ in range(100):
                    big.add_(1.0)
                done = torch.cuda.Event()
                done.record()
            time.sleep(0.001)
            start = time.perf_counter()
            plan.run(0.85, 20, out=out)
            main.synchronize()
            times.append(time.perf_counter() - start)
            assert not done.query()  # the other stream was busy all the while
        median[places] = sorted(times)[4]
    torch.cuda.synchronize()
    plan.close()
    assert median[64] < median[1] / 3


def test_infinite_degrees_stay_in_the_ranks():
    """A NaN and an infinity among the inverse out-degrees reach the ranks that they reach by way of row blocks."""
    import torch
    from drone_amd.pagerank import PullPlanF64
    rp, ci, inv = _matrix(500, [], 2)
    inv[3], inv[4] = np.nan, np.inf
    plan = _plan(rp, ci, inv)
    blocks = PullPlanF64(*(torch.from_numpy(a).cuda() for a in (rp, ci, inv)), shared_blocks=False)
    for iters in (1, 3):
        got = plan.run(0.85, iters).cpu().numpy()
        want = blocks.run(0.85, iters).cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        there = np.isfinite(want)
        assert (iters > 1 or there.any()) and np.allclose(got[there], want[there], rtol=1e-13, atol=0)
    plan.close()
    blocks.close()


def test_replays_of_a_recorded_run():
    import torch
    from drone_amd.pagerank import PullPlanF64
    rp, ci, inv = (torch.from_numpy(a).cuda() for a in _matrix(5000, [900, 1500], 9))
    side = torch.cuda.Stream()
    plan = PullPlanF64(rp, ci, inv)
    eager = plan.run(0.85, 7)
    torch.cuda.synchronize()
    plan.stream = side.cuda_stream
    out, graph = torch.zeros_like(eager), torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        plan.run(0.85, 7, out=out)
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            plan.run(0.85, 7, out=out)
    for _ in range(4):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    plan.close()


def test_runs_beside_each_other():
    """Four plans on four streams, whose work-groups ask for places at the same time."""
    import torch
    from drone_amd.pagerank import PullPlanF64
    mats = [[torch.from_numpy(a).cuda() for a in _matrix(n, [900], 9)] for n in (3000, 5000, 7000, 9000)]
    plans = [PullPlanF64(*m) for m in mats]
    want = [p.run(0.85, 20) for p in plans]
    torch.cuda.synchronize()
    outs = [torch.zeros_like(w) for w in want]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in plans]
    for p, s in zip(plans, streams):
        p.stream = s.cuda_stream
    for _ in range(50):
        for p, o in zip(plans, outs):
            p.run(0.85, 20, out=o)
    torch.cuda.synchronize()
    for p, o, w in zip(plans, outs, want):
        assert torch.equal(o, w)  # also where one run was a work-group's alone
        p.close()


def test_plans_that_share_a_kernel(oracle):
    """Plans of 1,024 rows with entries each: their runs are one kernel, which asks for 152, 8 and 40 KB of LDS in turn."""
    plans = []
    for rest in (9000, 0, 2000):
        rp, ci, inv = _matrix(1024 + rest, [5] * 1024, 0)
        plans.append((_plan(rp, ci, inv), oracle.pr_pull_f64(rp, ci, inv, 0.85, 6), rp))
    for plan, want, rp in plans:
        _close(plan.run(0.85, 6).cpu().numpy(), want, rp, 6)
    for plan, _, _ in plans:
        plan.close()


@pytest.mark.parametrize("iters", [2, 3, 20])
def test_profiled_runs_are_the_same_runs(iters):
    import torch
    plan = _plan(*_matrix(4097, [800] * 30, 11))
    want = plan.run(0.85, iters)
    plan.profile_enable(64)
    begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    begin.record()
    for _ in range(3):
        assert torch.equal(plan.run(0.85, iters), want)
    end.record()
    torch.cuda.synchronize()
    prof = plan.profile_read()
    assert prof["launches"] == 3 * iters and 0 < prof["min_ms"] <= prof["mean_ms"] <= prof["max_ms"]
    assert prof["mean_ms"] * 3 * iters <= begin.elapsed_time(end)
    assert plan.profile_read()["launches"] == 0
    plan.profile_enable(1)                               # fewer pairs of events than launches
    for _ in range(2):
        assert torch.equal(plan.run(0.85, iters), want)
    assert plan.profile_read()["launches"] == (iters if iters >= 3 else 1)
    plan.profile_enable(0)
    plan.close()


@pytest.mark.parametrize("n,shortest", [(10240, 3), (10241, 8), (12288, 8)])
def test_short_runs_that_would_wait_for_empty_cus_are_a_launch_per_iteration(n, shortest):
    """With one pair of events a run in one launch counts all its iterations, and a launch per iteration the first."""
    plan = _plan(*_matrix(n, [], 9))
    for iters in (shortest - 1, shortest):
        plan.profile_enable(1)
        plan.run(0.85, iters)
        assert plan.profile_read()["launches"] == (iters if iters == shortest else 1)
    plan.close()
