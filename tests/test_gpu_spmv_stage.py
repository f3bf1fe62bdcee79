"""The staged CSR products of ffhip_spmv (A x, A' x, half storage) at the sizes
where the staging can go wrong: 64-row blocks and their remainders, empty rows,
rows and blocks longer than the stage.

Bar: |y - y64| <= 2 (L + 2) u sum |a x| per row (L the row length, u = 2^-53),
the bound of one fused pass over a row on each side.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


def symmetric_pattern(n, spread, dense, seed):
    """symmetric pattern, random values: a random band, `dense` full rows and
    columns, every fifth row empty off them"""
    rng = np.random.default_rng(seed)
    M = np.zeros((n, n), bool)
    for i in range(n):
        if i % 5 != 4:
            j = i + rng.integers(-spread, spread + 1, 9)
            j = j[(j >= 0) & (j < n) & (j % 5 != 4)]
            M[i, j] = M[j, i] = True
            M[i, i] = True
    for d in range(dense):
        i = (7 * d + 3) % n
        M[i, :] = M[:, i] = True
    rows, ci = np.nonzero(M)
    rp = np.concatenate([[0], np.cumsum(M.sum(1))]).astype(np.int64)
    return rp, ci.astype(np.int32), rows, rng.standard_normal(rows.size)


def close(y, n, r, c, v, x):
    s = np.zeros(n, np.longdouble)
    m = np.zeros(n)
    np.add.at(s, r, v.astype(np.longdouble) * x[c])
    np.add.at(m, r, np.abs(v * x[c]))
    L = np.bincount(r, minlength=n)
    assert (np.abs(y - s) <= 2 * (L + 2) * 2.0 ** -53 * m).all()


@pytest.mark.parametrize("n,spread,dense", [(1, 1, 0), (63, 4, 0), (64, 30, 0), (65, 5, 1), (257, 40, 0),
                                            (1100, 60, 2), (2050, 200, 1), (4096, 12, 0)])
def test_products(n, spread, dense):
    import torch
    rp, ci, rows, v = symmetric_pattern(n, spread, dense, n)
    if rows.size == 0:
        pytest.skip("empty matrix")
    A = ffhip.Matrix.upload(rp, ci, v)
    x = np.random.default_rng(1).standard_normal(n)
    xd = torch.tensor(x, device="cuda")
    y = torch.full_like(xd, float("nan"))
    A.spmv(xd, y)
    close(y.cpu().numpy(), n, rows, ci, v, x)
    A.spmv(xd, y, trans=True)
    close(y.cpu().numpy(), n, ci, rows, v, x)
    low = ci <= rows
    rl = np.concatenate([[0], np.cumsum(np.bincount(rows[low], minlength=n))]).astype(np.int64)
    L = ffhip.Matrix.upload(rl, ci[low], v[low])
    L.set_half(1)
    L.spmv(xd, y)
    off = low & (ci < rows)
    close(y.cpu().numpy(), n, np.concatenate([rows[low], ci[off]]), np.concatenate([ci[low], rows[off]]),
          np.concatenate([v[low], v[off]]), x)


def test_transpose_of_unsymmetric_pattern_is_refused():
    import torch
    rp = np.array([0, 2, 3], np.int64)
    A = ffhip.Matrix.upload(rp, np.array([0, 1, 1], np.int32), np.array([1., 2., 3.]))
    x = torch.ones(2, dtype=torch.float64, device="cuda")
    with pytest.raises(ffhip.FFHipError) as e:
        A.spmv(x, torch.empty_like(x), trans=True)
    assert e.value.code == -5
