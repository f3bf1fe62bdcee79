"""FP64 solves of small systems in one workgroup: at the edges of a slice (64
rows), of a block (256), of a wave's turns (1024) and of the range (4096; in CSR 256), with
rows past the 16 entries of one round, Dirichlet rows, a transposed and a
capped solve.  The sums are those of the kernel-by-kernel launches
(graph=False): the bits must be the same.  Against the oracle: the CG tests'
bars."""
import numpy as np
import pytest

import ffo

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


def system(n, far, seed):
    """diagonally dominant symmetric band of offsets 1, 17 and, far, 20 more; every
    13th row a Dirichlet row (tgv)"""
    rng = np.random.default_rng(seed)
    M = {}
    for d in [1, 17] + (list(range(30, 50)) if far else []):
        for i in range(n - d):
            M[i, i + d] = M[i + d, i] = -rng.random()
    diag = np.ones(n) * 1e-2
    for (i, j), v in M.items():
        diag[i] -= v
    for i in range(n):
        M[i, i] = 1e30 if i % 13 == 5 else diag[i]
    keys = sorted(M)
    rp = np.concatenate([[0], np.cumsum(np.bincount([k[0] for k in keys], minlength=n))]).astype(np.int64)
    b = rng.standard_normal(n)
    b[5::13] *= 1e30
    return rp, np.array([k[1] for k in keys], np.int32), np.array([M[k] for k in keys]), b


@pytest.mark.parametrize("layout,n,far", [("sell", n, far) for n in (1, 2, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025,
                                                                    2000, 2048, 3900, 4095, 4096, 4097)
                                         for far in (False, True)] +
                         [("csr", n, False) for n in (1, 15, 16, 17, 64, 100, 127, 128, 129, 255, 256, 257)])
def test_one_workgroup_equals_launches(layout, n, far):
    rp, ci, va, b = system(n, far, n)
    A = ffhip.Matrix.upload(rp, ci, va)
    one, many = ffhip.CG(A, layout=layout), ffhip.CG(A, layout=layout, graph=False)
    assert one.layout()[0] == {"sell": "sell16", "csr": "csr"}[layout]
    for trans in (False, True):
        x, st = one.solve(b, eps=1e-10, trans=trans)
        xm, sm = many.solve(b, eps=1e-10, trans=trans)
        assert np.array_equal(x, xm)
        assert all(st[k] == sm[k] for k in ("iters", "converged", "gcg0", "gcg", "true_gcg", "true_relres"))
        xo, so = ffo.pcg(rp, ci, va, b, eps=1e-10, trans=trans)
        assert st["converged"] == 1 and abs(st["iters"] - so["iters"]) <= 1
        assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)
    for itmax in (1, 5):  # not converged, from a non-zero start
        x, st = one.solve(b, x=xo * 0.5, eps=1e-14, itmax=itmax, raise_on_error=False)
        xm, sm = many.solve(b, x=xo * 0.5, eps=1e-14, itmax=itmax, raise_on_error=False)
        assert np.array_equal(x, xm) and st["iters"] == sm["iters"] and st["converged"] == sm["converged"]


def test_device_vectors_zero_rhs_and_nan():
    import torch
    rp, ci, va, b = system(700, False, 3)
    A = ffhip.Matrix.upload(rp, ci, va)
    cg = ffhip.CG(A)
    xh, _ = cg.solve(b)
    buf = torch.zeros(1401, dtype=torch.float64, device="cuda")
    bd, xd = buf[:700], buf[701:]  # x at an odd address
    bd.copy_(torch.tensor(b))
    cg.solve(bd, x=xd)
    assert np.array_equal(xd.cpu().numpy(), xh)
    assert np.array_equal(bd.cpu().numpy(), b)
    x, st = cg.solve(np.zeros(700))
    assert st["converged"] == 2 and not x.any()
    with pytest.raises(ffhip.FFHipError) as e:
        cg.solve(np.full(700, np.nan))
    assert e.value.code == -4
