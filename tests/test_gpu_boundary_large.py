"""Boundary integrals on meshes of the sizes whose waves take more vertices:
squares of 32 and of 64 vertices a wave, a cube past 2^22 vertices; right-hand
sides against the oracle (bar of the boundary tests, 1e-13 of the largest
entry), matrices through their row sums, which are the right-hand side's
integrals."""
import numpy as np
import pytest

import ffo

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


def oracle_rhs(M, labels):
    d = M.download()
    mo = dict(nv=M.nv, nbe=M.nbe, blab=d["blab"])
    if M.dim == 2:
        mo.update(xy=d["xyz"], bedges=d["belems"], tris=d["elems"], nt=M.nt)
    else:
        mo.update(xyz=d["xyz"], btri=d["belems"], tets=d["elems"], nt=M.nt)
    b = np.zeros(M.nv)
    ffo.p1_boundary(mo, labels, ffo.COEF_SIN3, 0.0, b=b)
    return b


@pytest.mark.parametrize("size", [(33, 30), (1447, 1447), (1449, 1450)])  # 2^21 between the last two
def test_square(size):
    M = ffhip.square(*size)
    labels = (1, 2, 4)
    bo = oracle_rhs(M, labels)
    b = ffhip.rhs_p1_boundary(M, np.zeros(M.nv), labels, ffhip.COEF_SIN3)
    assert np.abs(b - bo).max() <= 1e-13 * np.abs(bo).max()
    A = ffhip.Matrix.p1(M)
    A.set_values(np.zeros(A.nnz))
    A.assemble_p1_boundary(labels, ffhip.COEF_SIN3)
    rp, _, va = A.download()
    assert np.abs(np.add.reduceat(va, rp[:-1]) - bo).max() <= 1e-13 * np.abs(bo).max()


@pytest.mark.parametrize("size", [(150, 160, 171), (150, 160, 173)])  # 2^22 between them
def test_cube(size):
    M = ffhip.cube(*size)
    bo = oracle_rhs(M, (1, 4, 6))
    b = ffhip.rhs_p1_boundary(M, np.zeros(M.nv), (1, 4, 6), ffhip.COEF_SIN3)
    assert np.abs(b - bo).max() <= 1e-13 * np.abs(bo).max()
