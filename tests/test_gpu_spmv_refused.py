"""A' x of a pattern that is not symmetric is refused and y is left as it was."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


@pytest.mark.parametrize("n", [2, 65, 1100, 300000])  # a wave's rows, both numbers of rows per wave
def test_y_is_untouched(n):
    import torch
    rng = np.random.default_rng(n)
    diag = np.arange(n)
    rows = np.concatenate([diag, diag[:-1], diag[1:-1]])
    ci = np.concatenate([diag, diag[:-1] + 1, diag[1:-1] - 1])  # the last row lacks its entry left of the diagonal
    o = np.lexsort((ci, rows))
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    A = ffhip.Matrix.upload(rp, ci[o].astype(np.int32), rng.standard_normal(rows.size))
    x = torch.tensor(rng.standard_normal(n), device="cuda")
    y = torch.tensor(rng.standard_normal(n), device="cuda")
    before = y.clone()
    with pytest.raises(ffhip.FFHipError) as e:
        A.spmv(x, y, trans=True)
    assert e.value.code == -5
    assert torch.equal(y, before)
