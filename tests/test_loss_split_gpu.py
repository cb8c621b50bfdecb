"""The loss that chooses its truth from split and label: the same report and gradient, bit for bit, as the pass over the chosen truth, and
the truth written for every row; classes on either side of a lane's four, rows around a work-group's share, splits nobody is in."""
import ctypes as C

import numpy as np
import pytest

from test_loss_pass_gpu import Pass

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,classes,which", [(1, 1, 1), (127, 4, 2), (129, 16, 1), (65, 17, 3), (1000, 64, 1), (33, 65, 2), (40, 300, 1),
                                             (16_385, 200, 1), (300_001, 7, 2), (2_708, 7, 0)])
def test_loss_on_a_split(n, classes, which):
    import torch
    from drone_amd._lib import check, lib
    rng = np.random.default_rng(n + classes)
    z = torch.from_numpy(rng.standard_normal((n, classes + 1)).astype(np.float32)).cuda()
    label = torch.from_numpy(rng.integers(-1, classes + 1, n).astype(np.int32)).cuda()  # unlabelled and outside the classes too
    split = torch.from_numpy(rng.integers(1, 3, n).astype(np.int32)).cuda()  # 1 or 2: nobody is in 0 and 3
    want_truth = torch.where(split == which, label, torch.full_like(label, -1))
    truth = torch.full_like(label, 99)

    def run(chosen):
        grad, report = torch.full((n, classes), 5.0, device="cuda"), torch.zeros(5, dtype=torch.int32, device="cuda")
        p = Pass(n=n, classes=classes, logits=z.data_ptr(), ld=classes + 1, truth=None if chosen else want_truth.data_ptr(),
                 grad=grad.data_ptr(), ldg=classes, grad_scale=0.5, report=report.data_ptr())
        if chosen:
            check(lib().drone_loss_pass_split_f32(C.byref(p), split.data_ptr(), label.data_ptr(), which, truth.data_ptr(), None))
        else:
            check(lib().drone_loss_pass_f32(C.byref(p), None))
        torch.cuda.synchronize()
        return grad, report

    for a, b in zip(run(False), run(True)):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    assert torch.equal(truth, want_truth)


def test_loss_on_a_split_refuses():
    import torch
    from drone_amd._lib import lib
    x = torch.zeros(8, device="cuda")
    p, at = Pass(n=2, classes=2, logits=x.data_ptr(), ld=2), x.data_ptr()
    for args in ((None, at, at), (at, None, at), (at, at, None)):
        assert lib().drone_loss_pass_split_f32(C.byref(p), args[0], args[1], 1, args[2], None) == -1
    assert lib().drone_loss_pass_f32(C.byref(p), None) == -1  # without a split it needs the truth


def test_epochs_leave_the_truth_of_their_split():
    """train_epoch() and eval() in turn, sum- and mean-reduced: the truth that a program reads afterwards is their split's, and the
    weights are those of set_truth() and the step."""
    import torch
    from drone_amd import gcn
    n, rng = 500, np.random.default_rng(3)
    rp = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    ci = torch.arange(n, dtype=torch.int32, device="cuda")
    one = torch.ones(n, dtype=torch.int32, device="cuda")
    X = torch.from_numpy(rng.standard_normal((n, 12)).astype(np.float32)).cuda()
    label = torch.from_numpy(rng.integers(0, 5, n).astype(np.int32)).cuda()
    split = torch.from_numpy(rng.integers(1, 4, n).astype(np.int32)).cuda()
    W1, W2 = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda() for s in ((12, 8), (8, 5)))
    for mean in (False, True):
        a, b = (gcn.GcnModel(rp, ci, one, one, X, label, split, W1, W2, use_adam=False, lr=0.01, mean_gradient=mean) for _ in range(2))
        for which in (1, 2, 1, 3, 1):
            if which == 1:
                a.train_epoch()
                b.set_truth(1)
                b.train_step_async()
            else:
                a.eval(which)
                b.set_truth(which)
                b.forward(False)
            torch.cuda.synchronize()
            np.testing.assert_array_equal(a.tensor("truth"), np.where(split.cpu().numpy() == which, label.cpu().numpy(), -1))
            np.testing.assert_array_equal(a.tensor("truth"), b.tensor("truth"))
            for name in ("W1", "W2"):
                np.testing.assert_array_equal(a.tensor(name), b.tensor(name))
        a.close(), b.close()
