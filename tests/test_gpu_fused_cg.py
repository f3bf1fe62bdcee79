"""Systems past one workgroup's size form the direction in the mat-vec, up to
327680 rows in FP64 and 2^20 in FP32: just past the smallest, in every layout,
transposed, stopped at an iteration cap (the last step is the stopping launch's)
against the oracle, and on both sides of the FP64 limit FP64 against MIXED.
Bars of the CG tests: iterations within 1, x within 1e-8."""
import numpy as np
import pytest

import ffo

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


@pytest.fixture(scope="module")
def system():
    return ffo.poisson_p1_3d(17)  # 5832 rows


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("layout,name", [("sell", "sell16"), ("sell32", "sell"), ("csr", "csr")])
@pytest.mark.parametrize("mode", [0, 1])
def test_against_oracle(system, mode, layout, name, trans):
    m, rp, ci, va, on, b = system
    xo, so = ffo.pcg(rp, ci, va, b, eps=1e-10, trans=trans)
    sols = []
    for graph in (True, False):
        cg = ffhip.CG(ffhip.Matrix.upload(rp, ci, va), mode, layout=layout, graph=graph)
        assert cg.layout()[0] == name
        x, st = cg.solve(b, eps=1e-10, trans=trans)
        assert st["converged"] == 1
        if mode == ffhip.CG_FP64:
            assert abs(st["iters"] - so["iters"]) <= 1
        assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)
        sols.append(x)
    assert np.array_equal(*sols)


@pytest.mark.parametrize("itmax", [1, 2, 15, 16, 17, 31])
def test_cap(system, itmax):
    m, rp, ci, va, on, b = system
    x, st = ffhip.CG(ffhip.Matrix.upload(rp, ci, va)).solve(b, eps=1e-14, itmax=itmax, raise_on_error=False)
    xo, so = ffo.pcg(rp, ci, va, b, eps=1e-14, itmax=itmax)
    assert st["iters"] == itmax and st["converged"] == 0
    assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)


@pytest.mark.parametrize("n", [67, 68])  # 314432 and 328509 rows
def test_around_the_limit(n):
    M = ffhip.cube(n)
    A = ffhip.Matrix.p1_assembled(M, ffhip.COEF_SIN3)
    labels = (1, 2, 3, 4, 5, 6)
    A.set_bc(labels)
    b = ffhip.rhs_p1(M, 1.0, labels)
    x, s = ffhip.CG(A).solve(b, eps=1e-10)
    y, t = ffhip.CG(A, ffhip.CG_MIXED).solve(b, eps=1e-10)
    assert s["converged"] == t["converged"] == 1
    assert np.linalg.norm(x - y) <= 1e-8 * np.linalg.norm(y)
