"""The 3x3-block products on both sides of the rule that shares a slice among a
block's waves: 2894 slices (fewer than the waves), 3547 (more: a wave per slice;
the FP32 copy of 3209 slices is still shared, it stays in the caches).  Against
the CSR product in FP64; bar 2 (L + 2) u sum |a x| per row, L the row length."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


@pytest.mark.parametrize("n", [2, 28, 29, 30])
def test_products(n):
    import torch
    S = ffhip.P2VSpace(ffhip.cube(n))
    A = ffhip.Matrix.p2v(S)
    A.assemble_p2v_elasticity(1.2, 0.7)
    cg = ffhip.CG(A, ffhip.CG_MIXED)
    assert cg.layout()[0] == "bsr3"
    rp, ci, va = A.download()
    L = int(np.diff(rp).max())
    d = torch.tensor(va[rp[:-1] + np.array([np.searchsorted(ci[a:b], i) for i, (a, b) in
                                            enumerate(zip(rp[:-1], rp[1:]))])], device="cuda")
    g = torch.Generator().manual_seed(n)
    x = torch.randn(A.n, generator=g, dtype=torch.float64).cuda()
    M = ffhip.Matrix.upload(rp, ci, np.abs(va))
    bound = torch.empty_like(x)
    y, z = torch.empty_like(x), torch.full_like(x, float("nan"))
    A.spmv(x, y)
    M.spmv(x.abs(), bound)
    for solver in (cg, ffhip.CG(A)):  # grids for three and for two blocks per CU
        solver.bench_spmv(0, 1, x, z)
        assert ((z - y).abs() <= 2 * (L + 2) * 2.0 ** -53 * bound).all()
        z.fill_(float("nan"))
    s = d.rsqrt()  # the FP32 copy holds D^-1/2 A D^-1/2
    x32, z32 = x.float(), torch.full_like(x, float("nan"), dtype=torch.float32)
    cg.bench_spmv(1, 1, x32, z32)
    xs = x32.double() * s
    A.spmv(xs, y)
    M.spmv(xs.abs(), bound)
    assert ((z32.double() - y * s).abs() <= 2 * (L + 2) * 2.0 ** -24 * bound * s).all()
