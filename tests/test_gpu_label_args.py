"""Boundary labels reach the kernels by value up to 16 and in an array beyond:
the marks, right-hand sides, boundary terms and the adjoint right-hand side are
the same, bit for bit, when labels that no boundary element has fill the list."""
import numpy as np
import pytest

import ffo

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


@pytest.mark.parametrize("count", [2, 15, 16, 17, 40])
def test_label_counts(count):
    import torch
    M, mo = ffhip.cube(5, 4, 3), ffo.cube(5, 4, 3)
    some = (1, 4)
    many = [100 + k for k in range(count - 2)] + list(some)
    ends = []
    for labels in (some, many):
        A = ffhip.Matrix.p1(M)
        A.assemble_p1(ffhip.COEF_SIN3)
        on = A.set_bc(labels, want_onbc=True)
        b = ffhip.rhs_p1(M, 1.5, labels, 1e30, 0.25)
        A.assemble_p1_boundary(labels, ffhip.COEF_CONST, 0.5)
        ffhip.rhs_p1_boundary(M, b, labels, ffhip.COEF_CONST, 0.7,
                              dirichlet=(2,) if labels == some else [200 + k for k in range(count)] + [2])
        g = torch.Generator(device="cuda").manual_seed(5)
        u, ud = (torch.randn(M.nv, generator=g, dtype=torch.float64, device="cuda") for _ in range(2))
        J, r = ffhip.p1_misfit(M, u, ud, labels)
        ends.append((on, A.download()[2], b, J, r.cpu().numpy()))
    want = ffo.mark_bc(mo["nv"], mo["btri"], mo["blab"], 3, some)
    assert np.array_equal(ends[0][0], want)
    for a, c in zip(*ends):
        assert np.array_equal(a, c)
