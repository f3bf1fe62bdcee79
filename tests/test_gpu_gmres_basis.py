"""GMRES over bases of more than one wave of vectors (64), of more than one
sweep of the coefficient solve (1024), batches cut by the restart and by the
iteration cap, and systems of fewer rows than a block; against the oracle's
fgmres.  Bars as in the GMRES tests: iterations within 1 (2 past 512
vectors), x within 1e-8."""
import numpy as np
import pytest

import ffo

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


def banded(n, seed, shift):
    """shift > 1: a rotation-like band; below, a cyclic shift with a diagonal,
    its eigenvalues around the origin: GMRES needs all n vectors"""
    rng = np.random.default_rng(seed)
    M = np.zeros((n, n))
    i = np.arange(n)
    M[i, i] = shift + 0.05 * rng.standard_normal(n)
    if shift > 1:
        M[i[:-1], i[:-1] + 1] = 1.0
        M[i[1:], i[1:] - 1] = -0.9
    else:
        M[i, (i + 1) % n] = 1.0
    rows, ci = np.nonzero(M)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    return rp, ci.astype(np.int32), M[rows, ci], rng.standard_normal(n)


@pytest.mark.parametrize("n,restart,shift,slack", [(3, 10, 1.5, 1), (64, 1000, 0.3, 1), (70, 1000, 0.3, 1),
                                                   (300, 7, 1.5, 1), (560, 1000, 0.3, 2), (1100, 1300, 0.3, 2)])
def test_gmres_basis(n, restart, shift, slack):
    rp, ci, va, b = banded(n, n, shift)
    cg = ffhip.CG(ffhip.Matrix.upload(rp, ci, va))
    for _ in range(2):  # the second solve on the kept basis
        x, st = cg.gmres(b, eps=1e-10, restart=restart)
        xo, so = ffo.fgmres(rp, ci, va, b, eps=1e-10, restart=restart)
        assert st["converged"] == so["converged"] == 1
        assert abs(st["iters"] - so["iters"]) <= slack, (st["iters"], so["iters"])
        assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)


@pytest.mark.parametrize("itmax", [1, 3, 4, 6])
def test_cap_inside_a_batch(itmax):
    rp, ci, va, b = banded(120, 5, 1.2)
    cg = ffhip.CG(ffhip.Matrix.upload(rp, ci, va))
    x, st = cg.gmres(b, eps=1e-12, itmax=itmax, restart=5, raise_on_error=False)
    xo, so = ffo.fgmres(rp, ci, va, b, eps=1e-12, itmax=itmax, restart=5)
    assert st["converged"] == so["converged"] == 0
    assert st["iters"] == so["iters"] and st["refinements"] == so["restarts"]
    assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)
