"""ReLU where it goes four elements at a time and where it may not (counts, addresses, special values), the optimisers over one to
four tensors, and the clearing of mirror rows around the rows a wavefront looks at together."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,x_off,mask_off", [(1, 0, 0), (3, 0, 0), (4, 0, 0), (1020, 0, 0), (1021, 0, 0), (1024, 1, 0), (1024, 0, 1),
                                              (1024, 2, 2), (1028, 4, 4), (262_148, 0, 0), (1_000_003, 3, 1), (4_200_000, 0, 0)])
def test_relu_at_every_alignment(n, x_off, mask_off):
    import torch
    from drone_amd import gcn
    rng = np.random.default_rng(n + x_off)
    values = rng.standard_normal(n).astype(np.float32)
    special = np.array([0.0, -0.0, np.nan, np.inf, -np.inf, 1e-45, -1e-45], np.float32)
    values[rng.integers(0, n, min(n, 50))] = rng.choice(special, min(n, 50))
    grads = rng.standard_normal(n).astype(np.float32)
    keep = values > 0
    for training in (True, False):
        x = torch.full((n + x_off + 4,), 9.0, device="cuda")
        mask = torch.full((n + mask_off + 4,), 7, dtype=torch.uint8, device="cuda")
        x[x_off:x_off + n] = torch.from_numpy(values)
        gcn.relu_forward(x[x_off:x_off + n], mask[mask_off:mask_off + n], training)
        got = x.cpu().numpy()
        np.testing.assert_array_equal(got[x_off:x_off + n].view(np.int32), np.where(keep, values, np.float32(0)).view(np.int32))
        assert (got[:x_off] == 9.0).all() and (got[x_off + n:] == 9.0).all()
        m = mask.cpu().numpy()
        np.testing.assert_array_equal(m[mask_off:mask_off + n], keep if training else np.full(n, 7))
        assert (m[:mask_off] == 7).all() and (m[mask_off + n:] == 7).all()
    x[x_off:x_off + n] = torch.from_numpy(grads)
    mask[mask_off:mask_off + n] = torch.from_numpy(keep.astype(np.uint8) * 3)  # any nonzero byte keeps
    gcn.relu_backward(x[x_off:x_off + n], mask[mask_off:mask_off + n])
    got = x.cpu().numpy()
    np.testing.assert_array_equal(got[x_off:x_off + n], np.where(keep, grads, 0))
    assert (got[:x_off] == 9.0).all() and (got[x_off + n:] == 9.0).all()


class Step(C.Structure):
    _fields_ = [("w", C.c_void_p), ("grad", C.c_void_p), ("m", C.c_void_p), ("v", C.c_void_p), ("n", C.c_int64), ("decay", C.c_int)]


@pytest.mark.parametrize("sizes", [(1,), (0, 5), (70_001, 64, 1_000_003), (255, 256, 257, 0)])
def test_optimiser_steps_over_several_tensors(oracle, sizes):
    import torch
    from drone_amd._lib import check, lib
    rng = np.random.default_rng(sum(sizes))
    for adam in (False, True):
        host = [[rng.standard_normal(n).astype(np.float32) for _ in range(4)] for n in sizes]
        for h in host:
            h[3] = np.abs(h[3])
        dev = [[torch.from_numpy(a.copy()).cuda() for a in h] for h in host]
        steps = (Step * len(sizes))(*[Step(*(t.data_ptr() if t.numel() else None for t in d), n, i % 2)
                                      for i, (d, n) in enumerate(zip(dev, sizes))])
        if adam:
            check(lib().drone_adam_steps_f32(steps, len(sizes), 5e-4, 0.01, 0.9, 0.999, 1e-8, 3, None))
        else:
            check(lib().drone_sgd_steps_f32(steps, len(sizes), 0.01, None))
        torch.cuda.synchronize()
        for i, (h, d) in enumerate(zip(host, dev)):
            w, g, m, v = h
            if adam and len(w):
                oracle.adam_step(w, g, m, v, bool(i % 2), 5e-4, 0.01, 0.9, 0.999, 1e-8, 3)
            elif len(w):
                oracle.sgd_step(w, g, 0.01)
            # a handful of fp32 roundings of values up to about 5
            for want, got in zip((w, m, v) if adam else (w,), (d[0], d[2], d[3]) if adam else (d[0],)):
                np.testing.assert_allclose(got.cpu().numpy(), want, rtol=1e-6, atol=2e-6)
            np.testing.assert_array_equal(d[1].cpu().numpy(), g)


@pytest.mark.parametrize("rows,K,ld", [(1, 1, 1), (15, 64, 64), (16, 65, 70), (17, 3, 3), (1023, 50, 52), (70_001, 1, 4), (1_100_003, 2, 2)])
def test_clear_mirror_rows_at_the_edges_of_a_wavefront(rows, K, ld):
    import torch
    from drone_amd import gcn
    rng = np.random.default_rng(rows)
    full = torch.from_numpy(rng.standard_normal((rows, ld)).astype(np.float32)).cuda()
    m2w = np.where(rng.random(rows) < 0.4, rng.integers(0, 4, rows), -1).astype(np.int32)
    m2w[-1] = 2
    want = full.cpu().numpy().copy()
    want[m2w != -1, :K] = 0.0
    gcn.clear_mirror_rows(full[:, :K], torch.from_numpy(m2w).cuda())
    np.testing.assert_array_equal(full.cpu().numpy(), want)
