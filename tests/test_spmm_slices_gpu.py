"""The aggregation at every width of its lane groups and slices, at any alignment: feature widths around powers of two, operands whose
rows start off 16-byte and 128-byte boundaries or lie in a wider array, operands below and above the size from which slices go by whole
lines (32 MB), few and many wavefronts, and plans that keep a part as bits."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

#        feature widths, leading dimensions, first column, rows, columns, entries a row
CASES = {
    "narrow": ([1, 2, 3, 4, 5, 6, 7, 8, 9], [9, 12, 13], 1, 301, 401, 9),
    "groups": ([15, 16, 17, 31, 32, 33, 63, 64, 65, 66], [67, 68], 0, 301, 401, 30),
    "few_wavefronts": ([100, 127, 128, 129, 160, 255, 256, 257, 300], [300, 301], 3, 301, 401, 300),
    "many_wavefronts": ([10, 61, 97, 128], [128, 131], 0, 12_001, 20_011, 40),
    "lines": ([97, 111, 112, 113, 125, 128], [128, 160], 0, 4_001, 90_001, 40),
    "no_lines": ([113, 128], [132, 129], 0, 4_001, 90_001, 40),
    "four_slices": ([239, 240, 241, 254, 256], [256], 0, 3_001, 40_001, 40),
}


def _check_sums(got, want, magnitude, lengths, at):
    """magnitude: sums of the terms' magnitudes.  A sum of d terms takes at most d + 12 roundings of 2^-24 of that (the products are fused;
    6 folds of lanes, 3 for the scalings, 3 to spare), in the worst case in one direction.  Over many sums they do not: partial sums of k random
    signs are about sqrt(k) of a term, so the roundings of a sum add up to sqrt(1 + 2 + ... + d) of 2^-24 / sqrt(3) of a term, at most
    0.6 of 2^-24 of the d terms' magnitudes, whatever d; the root mean square is held to 1."""
    err = np.abs(got - want) / np.maximum(magnitude, 1e-30) * 2.0 ** 24
    assert np.max(err / (np.asarray(lengths)[:, None] + 12)) <= 1.0, at
    assert np.sqrt(np.mean(err ** 2)) <= 1.0, at


@pytest.mark.parametrize("name", CASES)
def test_every_width_and_alignment(name):
    import torch
    from drone_amd import gcn
    widths, lds, first, n_rows, n_cols, mean = CASES[name]
    rng = np.random.default_rng(len(name))
    lengths = rng.poisson(mean, n_rows)
    lengths[rng.integers(0, n_rows, 9)] = [0, 0, 1, 64, 65, 129, 512, 513, 1300]
    lengths = np.minimum(lengths, n_cols)
    indptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    # distinct columns of a row: a start, and steps that do not come round
    cols = np.concatenate([np.sort((int(rng.integers(n_cols)) + np.arange(d) * max(1, n_cols // max(d, 1))) % n_cols) for d in lengths])
    m = sp.csr_matrix((rng.uniform(-1, 1, indptr[-1]).astype(np.float32), cols.astype(np.int32), indptr), shape=(n_rows, n_cols))
    m64, mabs = m.astype(np.float64), abs(m).astype(np.float64)
    rp, ci, v = (torch.from_numpy(a).cuda() for a in (indptr, m.indices, m.data))
    for ld in lds:
        room = rng.uniform(-1, 1, n_cols * ld + first).astype(np.float32)
        C0 = rng.uniform(-1, 1, n_rows * ld + first).astype(np.float32)
        B = np.lib.stride_tricks.as_strided(room[first:], (n_cols, ld), (4 * ld, 4))
        Bd = torch.from_numpy(room).cuda()[first:].as_strided((n_cols, ld), (ld, 1))
        for K in (k for k in widths if k <= ld):
            plan = gcn.SpmmPlan(rp, ci, v, n_cols, max_k=K)
            want, scale = m64 @ B[:, :K].astype(np.float64), mabs @ np.abs(B[:, :K].astype(np.float64))
            for beta in (0.0, -0.5):
                whole = torch.from_numpy(C0.copy()).cuda()
                out = whole[first:].as_strided((n_rows, ld), (ld, 1))
                gcn.spmm(plan, rp, ci, v, Bd, K=K, out=out, alpha=1.5, beta=beta)
                got = whole.cpu().numpy()
                before = C0[first:].reshape(n_rows, ld)
                after = got[first:].reshape(n_rows, ld)
                np.testing.assert_array_equal(got[:first], C0[:first])
                np.testing.assert_array_equal(after[:, K:], before[:, K:])
                _check_sums(after[:, :K], 1.5 * want + beta * before[:, :K], 1.5 * scale + 0.5 * np.abs(before[:, :K]), lengths, (ld, K, beta))
            plan.close()


@pytest.mark.parametrize("K,ld", [(6, 7), (41, 41), (97, 99), (127, 128), (128, 128), (131, 131), (250, 251)])
def test_bits_at_any_alignment(monkeypatch, K, ld):
    """A pattern with a dense corner, kept as bits, whatever the alignment of the rows."""
    import torch
    from drone_amd import gcn
    monkeypatch.setenv("DRONE_SPMM_DENSE_MIN_GAIN_MS", "0")
    rng = np.random.default_rng(K)
    n = 5000
    dense = sp.random(1500, n, 0.25, format="csr", random_state=3)
    m = sp.vstack([dense, sp.random(n - 1500, n, 0.002, format="csr", random_state=4)]).tocsr()
    m.sort_indices()
    rows, colscale = rng.uniform(0.5, 1, n).astype(np.float32), rng.uniform(0.5, 1, n).astype(np.float32)
    val = (np.repeat(rows, np.diff(m.indptr)) * colscale[m.indices]).astype(np.float32)
    m = sp.csr_matrix((val, m.indices, m.indptr), shape=m.shape)
    rp, ci, v, rs, cs = (torch.from_numpy(np.ascontiguousarray(a)).cuda()
                         for a in (m.indptr.astype(np.int32), m.indices.astype(np.int32), m.data, rows, colscale))
    B, C0 = (rng.uniform(-1, 1, (n, ld)).astype(np.float32) for _ in range(2))
    Bd = torch.from_numpy(B).cuda()
    plan = gcn.SpmmPlan(rp, ci, v, n, max_k=K, row_scale=rs, col_scale=cs)
    assert plan.bit_core()["cells"] > 0
    m64 = m.astype(np.float64)
    want, scale = m64 @ B[:, :K].astype(np.float64), m64 @ np.abs(B[:, :K].astype(np.float64))
    for beta in (0.0, 2.0):
        out = torch.from_numpy(C0.copy()).cuda()
        gcn.spmm(plan, rp, ci, v, Bd, K=K, out=out, alpha=0.75, beta=beta)
        got = out.cpu().numpy()
        np.testing.assert_array_equal(got[:, K:], C0[:, K:])
        # (the three parts of an operand in the bit core add up to it exactly)
        _check_sums(got[:, :K], 0.75 * want + beta * C0[:, :K], 0.75 * scale + abs(beta) * np.abs(C0[:, :K]), np.diff(m.indptr), beta)
    plan.close()


def test_bits_of_fewer_columns_after_nan(monkeypatch):
    """Products of every width of the bit core's tiles behind one that left a NaN in every place of the plan's operand and partial sums:
    what a narrower product does not write it does not read."""
    import torch
    from drone_amd import gcn
    monkeypatch.setenv("DRONE_SPMM_DENSE_MIN_GAIN_MS", "0")
    rng = np.random.default_rng(8)
    n, most = 5000, 256
    m = sp.vstack([sp.random(1500, n, 0.25, format="csr", random_state=3), sp.random(n - 1500, n, 0.002, format="csr", random_state=4)]).tocsr()
    m.sort_indices()
    m.data[:] = 1.0
    m = m.astype(np.float32)
    ones = torch.ones(n, device="cuda")
    rp, ci, v = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (m.indptr.astype(np.int32), m.indices.astype(np.int32), m.data))
    B = rng.uniform(-1, 1, (n, most)).astype(np.float32)
    Bd, none = torch.from_numpy(B).cuda(), torch.full((n, most), np.nan, device="cuda")
    plan = gcn.SpmmPlan(rp, ci, v, n, max_k=most, row_scale=ones, col_scale=ones)
    assert plan.bit_core()["cells"] > 0
    m64 = m.astype(np.float64)
    want, scale = m64 @ B.astype(np.float64), m64 @ np.abs(B).astype(np.float64)
    out = torch.empty(n, most, device="cuda")
    for K in (1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 128, 129, 144, 145, 176, 192, 224, 225, 256):
        gcn.spmm(plan, rp, ci, v, none, K=most, out=out)
        torch.cuda.synchronize()
        assert bool(out[torch.from_numpy(np.diff(m.indptr) > 0).cuda()].isnan().all())
        gcn.spmm(plan, rp, ci, v, Bd, K=K, out=out)
        _check_sums(out.cpu().numpy()[:, :K], want[:, :K], scale[:, :K], np.diff(m.indptr), K)
    plan.close()


def test_pieces_join_their_rows_again_and_again():
    """One plan, products of several widths in turn, with and without what was there before: the rows' tickets start over each time."""
    import torch
    from drone_amd import gcn
    rng = np.random.default_rng(12)
    n_cols = 6000
    lengths = np.concatenate([rng.integers(0, 40, 500), [513, 640, 641, 1025, 5999, 6000, 700, 2049]])
    indptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    cols = np.concatenate([np.sort(rng.permutation(n_cols)[:d]) for d in lengths]).astype(np.int32)
    m = sp.csr_matrix((rng.uniform(-1, 1, indptr[-1]).astype(np.float32), cols, indptr), shape=(len(lengths), n_cols))
    rp, ci, v = (torch.from_numpy(a).cuda() for a in (indptr, m.indices, m.data))
    B = rng.uniform(-1, 1, (n_cols, 260)).astype(np.float32)
    Bd, C0 = torch.from_numpy(B).cuda(), torch.from_numpy(rng.uniform(-1, 1, (len(lengths), 260)).astype(np.float32)).cuda()
    plan = gcn.SpmmPlan(rp, ci, v, n_cols, max_k=260)
    want, scale = m.astype(np.float64) @ B.astype(np.float64), abs(m).astype(np.float64) @ np.abs(B.astype(np.float64))
    first = {}
    for turn in range(12):
        for K, beta in ((3, 0.0), (61, 1.0), (128, 0.0), (7, 1.0), (260, 0.0), (64, 1.0)):
            out = C0.clone()
            gcn.spmm(plan, rp, ci, v, Bd, K=K, out=out, beta=beta)
            if turn == 0:
                first[K] = out
                got, before = out.cpu().numpy(), C0.cpu().numpy()
                _check_sums(got[:, :K], (want + beta * before)[:, :K], (scale + np.abs(before))[:, :K], lengths, (K, beta))
                assert np.array_equal(got[:, K:], before[:, K:])
            assert torch.equal(out, first[K])
    plan.close()
