"""drone_loss_pass_f32 where its work-groups begin and end: classes around the lanes of a row, rows around a work-group's share and
past the most work-groups, weights of none to many work-groups, mirrors, and the mean over a device count."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Report(C.Structure):
    _fields_ = [("loss", C.c_float), ("sum_squares", C.c_float), ("labelled", C.c_int), ("correct", C.c_int), ("counted", C.c_int)]


class Pass(C.Structure):
    _fields_ = [("n", C.c_int), ("classes", C.c_int), ("logits", C.c_void_p), ("ld", C.c_int), ("truth", C.c_void_p),
                ("grad", C.c_void_p), ("ldg", C.c_int), ("grad_scale", C.c_float), ("mean_over", C.c_void_p), ("skip", C.c_void_p),
                ("weights", C.c_void_p), ("weight_count", C.c_int64), ("loss", C.c_void_p), ("labelled", C.c_void_p),
                ("report", C.c_void_p)]


@pytest.mark.parametrize("n,classes,weights", [(1, 1, 0), (127, 4, 1), (128, 16, 2047), (129, 5, 2048), (65, 17, 2049), (1000, 64, 131_073),
                                               (33, 65, 5), (40, 128, 300), (16_384, 129, 77), (16_385, 200, 200_000),
                                               (300_001, 7, 4096), (70_003, 41, 10)])
def test_loss_pass_edges(n, classes, weights):
    import torch
    from drone_amd._lib import check, lib
    rng = np.random.default_rng(n + classes)
    z = rng.standard_normal((n, classes + 3)).astype(np.float32)
    truth = rng.integers(-1, classes + 1, n).astype(np.int32)  # unlabelled, labelled, and a label outside the classes
    skip = np.where(rng.random(n) < 0.3, 1, -1).astype(np.int32)
    w = rng.standard_normal(max(weights, 1)).astype(np.float32)
    d = {k: torch.from_numpy(a).cuda() for k, a in dict(z=z, truth=truth, skip=skip, w=w).items()}
    grad = torch.full((n, classes + 2), 5.0, device="cuda")
    over, report = torch.tensor([17], dtype=torch.int32, device="cuda"), torch.zeros(5, dtype=torch.int32, device="cuda")
    p = Pass(n=n, classes=classes, logits=d["z"].data_ptr(), ld=classes + 3, truth=d["truth"].data_ptr(), grad=grad.data_ptr(),
             ldg=classes + 2, grad_scale=1.0, mean_over=over.data_ptr(), skip=d["skip"].data_ptr(), weights=d["w"].data_ptr(),
             weight_count=weights, report=report.data_ptr())
    for _ in range(2):  # the counters of the first launch are back at zero
        check(lib().drone_loss_pass_f32(C.byref(p), None))
    r = Report.from_buffer_copy(report.cpu().numpy().tobytes())
    x = z[:, :classes].astype(np.float64)
    labelled = (truth >= 0) & (truth < classes)
    t = np.where(labelled, truth, 0)
    zt, mx = x[np.arange(n), t], x.max(1)
    e = np.exp(x - mx[:, None])
    loss = np.log(e.sum(1)) - (zt - mx)
    counted = labelled & (skip == -1)
    assert (r.labelled, r.counted, r.correct) == (labelled.sum(), counted.sum(), (counted & (zt >= mx)).sum())
    # fp32 exp, log and sums of up to `classes` terms near 1: a few eps each, in a loss of at most about 10
    if labelled.any():
        assert abs(r.loss - loss[labelled].mean()) <= 1e-5
    assert abs(r.sum_squares - (w[:weights].astype(np.float64) ** 2).sum()) <= 1e-6 * max(1.0, float((w[:weights] ** 2).sum()))
    onehot = np.zeros_like(x)
    onehot[np.arange(n), t] = 1.0
    want = np.where(labelled[:, None], (e / e.sum(1, keepdims=True) - onehot) / 17, 0.0)
    got = grad.cpu().numpy()
    np.testing.assert_allclose(got[:, :classes], want, rtol=0, atol=2e-6 / 17 * 8)  # 8 roundings of values up to 1, over 17
    assert (got[:, classes:] == 5.0).all()
