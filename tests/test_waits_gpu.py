"""Calls that return what the GPU has counted wait for their stream in a way that the runtime takes note of: it holds the stream for idle
when they return, so that what the program does next, a copy of the results most of all, does not wait once more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _idle_after(calls):
    import torch
    stream = torch.cuda.default_stream()  # the handles' own
    busy = []
    for name, call in calls:
        for i in range(40):
            call()
            if not stream.query():
                busy.append((name, i))
            torch.cuda.synchronize()
    assert not busy


def test_supersteps_leave_an_idle_stream():
    from drone_amd import pagerank
    rng = np.random.default_rng(5)
    n = 20_000
    w = pagerank.PRWorkerCUDA(n, rng.integers(0, n, 8 * n).astype(np.int32), np.arange(8 * n, dtype=np.int32) % n)
    w.peval()
    _idle_after([("peval", w.peval), ("incEval", w.incEval)])
    w.close()


def test_epochs_leave_an_idle_stream():
    import torch
    from drone_amd import gcn
    gen = torch.Generator(device="cuda").manual_seed(3)
    n, fin, hid, cls = 2000, 64, 16, 7
    key = torch.unique(torch.cat([torch.randint(0, n * n, (8 * n,), generator=gen, device="cuda"), torch.arange(n, device="cuda") * (n + 1)]))
    count = torch.bincount(key // n, minlength=n)
    rp = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    rp[1:] = torch.cumsum(count, 0)
    deg = count.to(torch.int32)
    label = torch.randint(0, cls, (n,), generator=gen, device="cuda", dtype=torch.int32)
    split = torch.where(torch.rand(n, generator=gen, device="cuda") < 0.66, 1, 2).to(torch.int32)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    model = gcn.GcnModel(rp, (key % n).to(torch.int32), deg, deg, draw(n, fin), label, split, draw(fin, hid), draw(hid, cls), use_adam=True, lr=0.01)
    _idle_after([("train_epoch", model.train_epoch), ("eval", lambda: model.eval(2))])
    model.close()
