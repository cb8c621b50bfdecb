"""Optimiser steps whose gradients are still the partial sums of a split reduction, and the products that leave them."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Tensor(C.Structure):
    _fields_ = [("w", C.c_void_p), ("grad", C.c_void_p), ("m", C.c_void_p), ("v", C.c_void_p), ("n", C.c_int64), ("decay", C.c_int)]


class Sums(C.Structure):
    _fields_ = [("sums", C.c_void_p), ("splits", C.c_int)]


@pytest.mark.parametrize("adam", [False, True])
@pytest.mark.parametrize("n,splits", [(1, 1), (31, 7), (32, 8), (33, 9), (448, 64), (8193, 65), (98304, 5), (0, 3)])
def test_steps_add_up_the_sums(n, splits, adam):
    import torch
    from drone_amd._lib import check, lib
    gen = torch.Generator(device="cuda").manual_seed(n + splits)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    parts = draw(splits, n)
    other = 1000                                    # a tensor whose gradient is there, in the same launch
    w, grad = [draw(n), draw(other)], [torch.full((n,), 7.0, device="cuda"), draw(other)]
    m, v = [draw(n), draw(other)], [draw(n).square(), draw(other).square()]
    before = [[x.double().cpu() for x in xs] for xs in (w, m, v)]
    given = grad[1].clone()
    t = (Tensor * 2)(*[Tensor(w[i].data_ptr(), grad[i].data_ptr(), m[i].data_ptr(), v[i].data_ptr(), w[i].numel(), i) for i in range(2)])
    s = (Sums * 2)(Sums(parts.data_ptr(), splits), Sums(None, 0))
    if adam:
        check(lib().drone_adam_steps_sums_f32(t, s, 2, 5e-4, 0.01, 0.9, 0.999, 1e-8, 3, None))
    else:
        check(lib().drone_sgd_steps_sums_f32(t, s, 2, 0.01, None))
    torch.cuda.synchronize()
    assert torch.equal(grad[1], given)
    exact = parts.double().sum(0)
    # a sum of `splits` terms in fp32 is within splits * 2^-24 of the sum of their magnitudes
    assert bool(((grad[0].double() - exact).abs() <= splits * 2.0 ** -24 * parts.double().abs().sum(0)).all())
    for i in range(2):
        W, M, V = (b[i] for b in before)
        g = grad[i].double().cpu()
        if adam:
            g = g + (5e-4 * W if i == 1 else 0.0)
            M, V = 0.9 * M + 0.1 * g, 0.999 * V + 0.001 * g * g
            step = 0.01 * np.sqrt(1 - 0.999 ** 3) / (1 - 0.9 ** 3)
            W = W - step * M / (V.sqrt() + 1e-8)
            # a handful of fp32 roundings each, and beta1, beta2 as floats: 1 - beta2 is good to 2^-24 / 1e-3
            assert torch.allclose(m[i].double().cpu(), M, rtol=1e-5, atol=1e-6) and torch.allclose(v[i].double().cpu(), V, rtol=1e-4, atol=1e-8)
            assert torch.allclose(w[i].double().cpu(), W, rtol=1e-5, atol=1e-4 * step * max(1.0, float((M / V.sqrt()).abs().max()) if W.numel() else 1.0))
        else:
            assert torch.allclose(w[i].double().cpu(), W - 0.01 * g, rtol=2.0 ** -22, atol=2.0 ** -24)


@pytest.mark.parametrize("M,N,K", [(1433, 64, 2708), (64, 7, 2708), (301, 100, 30011), (128, 41, 60000), (640, 128, 9000), (8, 5, 40)])
def test_products_leave_their_sums(M, N, K):
    """The sums of every kernel that splits its reduction add up to the product, and what does not split writes it."""
    import torch
    from drone_amd._lib import check, lib
    gen = torch.Generator(device="cuda").manual_seed(M)
    A, B = (torch.randn(K, c, generator=gen, device="cuda") for c in (M, N))
    want = (A.double().t() @ B.double())
    scale = (A.double().abs().t() @ B.double().abs())
    floats = lib().drone_sgemm_tn_sums_floats(M, N, K, M, N)
    for room in (floats, floats - 1):
        sums, out, splits = torch.full((max(floats, 1),), np.nan, device="cuda"), torch.full((M, N), np.nan, device="cuda"), C.c_int(-1)
        check(lib().drone_sgemm_tn_sums_f32(M, N, K, A.data_ptr(), M, B.data_ptr(), N, out.data_ptr(), N, sums.data_ptr(), room,
                                            C.byref(splits), None))
        torch.cuda.synchronize()
        if room > 0 and room == floats:
            assert splits.value * M * N == floats and splits.value > 1
            got = sums.view(splits.value, M, N).double().sum(0)
        else:
            assert splits.value == 0
            got = out.double()
        assert bool(((got - want).abs() <= K * 2.0 ** -24 * scale).all())  # K terms in fp32, in any order
