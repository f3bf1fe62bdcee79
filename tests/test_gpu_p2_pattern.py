"""P2 node rows around one pass of 64 candidates (6 elements), around 64 columns
(12 rings: 65), at the 96 the row buffers hold (18: 95) and past them (refused),
their vertices renumbered at random: patterns and slot maps (through the values)
against the oracle's.  Bars as in the P2 tests."""
import numpy as np
import pytest

import ffo
from test_gpu_p1 import _fan_mesh

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


def shuffled(m):
    mo = _fan_mesh(m)
    p = np.random.default_rng(m).permutation(mo["nv"]).astype(np.int32)
    X = np.empty_like(mo["xyz"].reshape(-1, 3))
    X[p] = mo["xyz"].reshape(-1, 3)
    return dict(mo, xyz=X.ravel().copy(), tets=p[mo["tets"]], btri=p[mo["btri"]])


@pytest.mark.parametrize("m", [3, 6, 7, 11, 12, 13, 18])
def test_pattern(m):
    mo = shuffled(m)
    sp = ffhip.P2VSpace(ffhip.mesh3_upload(mo["xyz"], mo["tets"], mo["btri"], mo["blab"]))
    q = ffo.poisson_p2(0, kind=ffo.COEF_CONST, c0=2.5, labels=(), mesh=mo)
    B = ffhip.Matrix.p2(sp)
    B.assemble_p2(ffhip.COEF_CONST, 2.5)
    rp, ci, va = B.download()
    assert np.array_equal(rp, q["rowptr"]) and np.array_equal(ci, q["colidx"])
    assert np.abs(va - q["vals"]).max() <= 1e-12 * np.abs(q["vals"]).max()
    A = ffhip.Matrix.p2v(sp)
    A.assemble_p2v_elasticity(1.7, 0.4)
    o = ffo.elasticity_p2(0, lam=1.7, mu=0.4, f=(0.3, -1.0, 2.0), labels=(), mesh=mo)
    rp, ci, va = A.download()
    assert np.array_equal(rp, o["rowptr"]) and np.array_equal(ci, o["colidx"])
    assert np.abs(va - o["vals"]).max() <= 1e-12 * np.abs(o["vals"]).max()
    for mode in (ffhip.CG_FP64, ffhip.CG_MIXED):  # slice widths, block slice widths
        for M in (A, B):
            assert ffhip.CG(M, mode).layout()[1] >= M.nnz


@pytest.mark.parametrize("m", [19, 33])
def test_too_many_columns(m):
    mo = shuffled(m)
    sp = ffhip.P2VSpace(ffhip.mesh3_upload(mo["xyz"], mo["tets"], mo["btri"], mo["blab"]))
    for make in (ffhip.Matrix.p2, ffhip.Matrix.p2v):
        with pytest.raises(ffhip.FFHipError) as e:
            make(sp)
        assert "more than 96 nodes" in str(e.value)
