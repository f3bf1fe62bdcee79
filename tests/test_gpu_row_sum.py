"""Right-hand sides and the adjoint's mass product at the sizes where the
staged row sums can go wrong: fewer than 64 rows, one row over, a last partial
block, and a vertex whose incidence list is longer than the stage.

Bar: 1e-13 of the largest entry (the right-hand side's bar in the cube tests).
"""
import numpy as np
import pytest

import ffo
from test_gpu_p1 import _fan_mesh

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")

MESHES = {"cube1": lambda: ffo.cube(1), "cube3": lambda: ffo.cube(3), "cube3x3x4": lambda: ffo.cube(3, 3, 4),
          "cube7x5x3": lambda: ffo.cube(7, 5, 3), "fan40": lambda: _fan_mesh(40), "fan1100": lambda: _fan_mesh(1100)}


@pytest.mark.parametrize("name", MESHES)
def test_row_sums(name):
    import torch
    mo = MESHES[name]()
    m = ffhip.mesh3_upload(mo["xyz"], mo["tets"], mo["btri"], mo["blab"])
    rng = np.random.default_rng(3)
    u, ud = rng.standard_normal(mo["nv"]), rng.standard_normal(mo["nv"])

    def close(a, b):
        assert np.abs(a - b).max() <= 1e-13 * np.abs(b).max()
    fe = rng.standard_normal(mo["nt"])
    close(ffhip.rhs_p1(m, 1.5), ffo.rhs_p1_coef(mo, ffo.COEF_CONST, 1.5))
    close(ffhip.rhs_p1_form(m, ffhip.COEF_P0, fcoef=fe), ffo.rhs_p1_coef(mo, ffo.COEF_P0, 0., fe))
    close(ffhip.rhs_p1_form(m, ffhip.COEF_SIN3), ffo.rhs_p1_coef(mo, ffo.COEF_SIN3))
    close(ffhip.rhs_p1_form(m, ffhip.COEF_P1, fcoef=u),
          ffo.rhs_p1_coef(mo, ffo.COEF_QP, 0., ffo.p1_at_qp(mo, u)))
    # J = e' M e / 2 and r = M e against the mass right-hand side of e = u - ud
    J, r = ffhip.p1_misfit(m, torch.tensor(u, device="cuda"), torch.tensor(ud, device="cuda"))
    Me = ffo.rhs_p1_coef(mo, ffo.COEF_QP, 0., ffo.p1_at_qp(mo, u - ud))
    close(r.cpu().numpy(), Me)
    assert abs(J - 0.5 * (u - ud) @ Me) <= 1e-12 * abs(J)
