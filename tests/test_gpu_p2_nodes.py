"""P2 assembly at node counts on both sides of each number of node rows per wave
(1 up to 4096 nodes, 2 up to 16384, 4 up to 100000, then 8), a part of a wave left
over, against the oracle.  Bar of the P2 tests: 1e-12 of the largest entry."""
import numpy as np
import pytest

import ffo

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")

BOXES = [(7, 7, 8), (8, 8, 8), (12, 12, 12), (12, 12, 14), (22, 22, 22), (22, 23, 24)]


@pytest.mark.parametrize("box", BOXES)
def test_scalar(box):
    mo = ffo.cube(*box)
    sp = ffhip.P2VSpace(ffhip.cube(*box))
    A = ffhip.Matrix.p2(sp)
    ke = np.exp(0.5 * np.random.default_rng(2).standard_normal(mo["nt"]))
    for kind, k in ((ffo.COEF_CONST, None), (ffo.COEF_SIN3, None), (ffo.COEF_P0, ke)):
        o = ffo.poisson_p2(0, kind=kind, c0=2.5, kappa_e=k, labels=(), mesh=mo)
        A.assemble_p2(kind, 2.5, k)
        va = A.download()[2]
        assert np.abs(va - o["vals"]).max() <= 1e-12 * np.abs(o["vals"]).max()


@pytest.mark.parametrize("box", BOXES[:4] + [(14, 14, 15), (22, 23, 24)])
def test_elasticity_rows_are_those_of_the_scalar_form(box):
    """lambda = 0, mu = 1: the trace over the components of a node block is
    4 times the scalar entry (mu (delta tr + transpose))"""
    sp = ffhip.P2VSpace(ffhip.cube(*box))
    A, B = ffhip.Matrix.p2v(sp), ffhip.Matrix.p2(sp)
    A.assemble_p2v_elasticity(0.0, 1.0)
    B.assemble_p2(ffhip.COEF_CONST, 1.0)
    rp, ci, va = A.download()
    rb, _, vb = B.download()
    L = np.diff(rb)
    # node a's rows 3a + c hold the blocks in order: entry 3 j + c of row c
    start = np.repeat(rp[0:-1:3], L) + 3 * (np.arange(rb[-1]) - np.repeat(rb[:-1], L))
    step = np.repeat(3 * L, L)
    tr = va[start] + va[start + step + 1] + va[start + 2 * step + 2]
    assert np.abs(tr - 4 * vb).max() <= 1e-12 * np.abs(vb).max()
