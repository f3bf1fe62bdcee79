"""GMRES launches as many iterations at a time as the solve seems to need: solves
that end in each of the first iterations, past the first batches, after a
restart, at once (a zero right-hand side, an exact start) and without progress,
against the oracle's fgmres.  Bars as in the GMRES tests: iterations within 1, x
within 1e-8 of the largest."""
import numpy as np
import pytest

import ffo

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


def system(n, shift):
    """tridiagonal, unsymmetric; the larger the shift the faster the solve"""
    rng = np.random.default_rng(n)
    M = np.diag(shift + 0.05 * rng.standard_normal(n)) + np.diag(np.ones(n - 1), 1) - 0.9 * np.diag(np.ones(n - 1), -1)
    rows, ci = np.nonzero(M)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    return rp, ci.astype(np.int32), M[rows, ci], rng.standard_normal(n)


@pytest.mark.parametrize("restart", [1000, 6])
@pytest.mark.parametrize("shift", [1e3, 30., 4.])
def test_first_iterations(shift, restart):
    rp, ci, va, b = system(300, shift)
    cg = ffhip.CG(ffhip.Matrix.upload(rp, ci, va))
    for eps in (0.5, 1e-1, 1e-2, 1e-3, 1e-4, 1e-6, 1e-9, 1e-12):
        x, st = cg.gmres(b, eps=eps, restart=restart, itmax=400)
        xo, so = ffo.fgmres(rp, ci, va, b, eps=eps, restart=restart, itmax=400)
        assert st["converged"] == so["converged"] == 1
        assert abs(st["iters"] - so["iters"]) <= 1, (eps, st["iters"], so["iters"])
        if st["iters"] == so["iters"]:
            assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)


def test_no_rest():
    rp, ci, va, b = system(300, 4.)
    cg = ffhip.CG(ffhip.Matrix.upload(rp, ci, va))
    x, _ = cg.gmres(b, eps=1e-13, raise_on_error=False)
    y, st = cg.gmres(b, x=x.copy(), eps=1e-6)  # the first residual is below the bar
    assert st["converged"] == 1 and st["iters"] <= 1
    assert np.linalg.norm(y - x) <= 1e-8 * np.linalg.norm(x)
    xo, so = ffo.fgmres(rp, ci, va, b, eps=0.0, itmax=9, restart=5)
    x, st = cg.gmres(b, eps=0.0, itmax=9, restart=5, raise_on_error=False)  # an eps that is never reached
    assert (st["iters"], st["converged"]) == (so["iters"], 0)
    assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)
