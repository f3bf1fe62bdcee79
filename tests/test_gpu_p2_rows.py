"""P2 node rows and right-hand sides at the sizes where the row kernels can go
wrong: one tet (fewer incidences than a group of six), rows of more than six
and of more than 12 incidences, node counts off the 8 and 64 rows of a wave,
irregular tets.  Bars as in the P2 tests: values 1e-12 of the largest entry,
right-hand sides 1e-14 (1e-13 on irregular tets)."""
import numpy as np
import pytest

import ffo
from test_gpu_p1 import _fan_mesh

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


def one_tet():
    return dict(nv=4, nt=1, nbe=4, xyz=np.array([0., 0, 0, 1.3, .1, 0, .2, .9, .1, .1, .3, 1.7]),
                tets=np.array([0, 1, 2, 3], np.int32), btri=np.array([3, 2, 1, 0, 2, 3, 3, 1, 0, 0, 1, 2], np.int32),
                blab=np.ones(4, np.int32))


def bent(m):
    X = m["xyz"].reshape(-1, 3)
    X = X + 0.06 * np.sin(3 * X[:, [1, 2, 0]] + 0.3)
    return dict(m, xyz=np.ascontiguousarray(X.ravel()))


MESHES = {"tet": one_tet, "fan4": lambda: _fan_mesh(4), "fan9": lambda: _fan_mesh(9),
          "box211": lambda: bent(ffo.cube(2, 1, 1)), "box345": lambda: bent(ffo.cube(3, 4, 5))}


@pytest.mark.parametrize("name", MESHES)
def test_rows(name):
    mo = MESHES[name]()
    sp = ffhip.P2VSpace(ffhip.mesh3_upload(mo["xyz"], mo["tets"], mo["btri"], mo["blab"]))
    o = ffo.elasticity_p2(0, lam=1.7, mu=0.4, f=(0.3, -1.0, 2.0), labels=(), mesh=mo)
    A = ffhip.Matrix.p2v(sp)
    A.assemble_p2v_elasticity(1.7, 0.4)
    rp, ci, va = A.download()
    assert np.array_equal(rp, o["rowptr"]) and np.array_equal(ci, o["colidx"])
    assert np.abs(va - o["vals"]).max() <= 1e-12 * np.abs(o["vals"]).max()
    b = ffhip.rhs_p2v(sp, (0.3, -1.0, 2.0))
    assert np.abs(b - o["b"]).max() <= 1e-13 * np.abs(o["b"]).max()
    for kind in (ffo.COEF_CONST, ffo.COEF_SIN3):
        q = ffo.poisson_p2(0, kind=kind, c0=2.5, labels=(), mesh=mo)
        B = ffhip.Matrix.p2(sp)
        B.assemble_p2(kind, 2.5)
        _, _, vb = B.download()
        assert np.abs(vb - q["vals"]).max() <= 1e-12 * np.abs(q["vals"]).max()
