"""Long FP64 solves of large box matrices read half of the values (the matrix
symmetric, its rows of few patterns): the same entries in the same order, so the
solution equals the transposed solve's (which reads all of them) bit for bit.
Matrices that lack the form (one entry an ulp off its mirror; rows of many
patterns) and new values keep to the other layout's solution (bar of the CG
tests: 1e-8)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")

BOXES = [(76, 77, 79), (64, 65, 130), (1200, 1100, 0)]  # 3D twice (a short plane), 2D


def system(box, kappa_seed=0):
    M = ffhip.cube(*box) if box[2] else ffhip.square(*box[:2])
    labels = (1, 2, 3, 4, 5, 6) if box[2] else (1, 2, 3, 4)
    A = ffhip.Matrix.p1(M)
    A.assemble_p1(ffhip.COEF_SIN3)
    A.set_bc(labels)
    return M, A, ffhip.rhs_p1(M, 1.0, labels)


def solve(cg, b, **kw):
    x, st = cg.solve(b, eps=1e-6, itmax=300, raise_on_error=False, **kw)
    assert st["iters"] > 64
    return x, st


@pytest.mark.parametrize("box", BOXES)
def test_half_equals_whole(box):
    M, A, b = system(box)
    for graph in (True, False):
        cg = ffhip.CG(A, layout="sell", graph=graph)
        assert cg.layout()[0] == "sell16"
        whole = solve(cg, b, trans=True)
        for _ in range(2):  # found in the first solve, used from the start in the second
            x, st = solve(cg, b)
            assert np.array_equal(x, whole[0]) and st["iters"] == whole[1]["iters"]
    A.assemble_p1(ffhip.COEF_CONST, 3.0)  # other values
    A.set_bc((1, 2, 3, 4, 5, 6) if box[2] else (1, 2, 3, 4))
    cg.update_values()
    assert np.array_equal(solve(cg, b)[0], solve(cg, b, trans=True)[0])


@pytest.mark.parametrize("what", ["ulp", "patterns"])
def test_other_matrices(what):
    _, A, b = system(BOXES[0])
    rp, ci, va = A.download()
    n = rp.size - 1
    if what == "ulp":
        rows = np.repeat(np.arange(n), np.diff(rp))
        k = np.flatnonzero((ci < rows) & (va < 0))[1000]
        va[k] = np.nextafter(va[k], -1)
    else:  # neighbours swapped at random
        rng = np.random.default_rng(1)
        p = np.arange(n)
        for i in np.flatnonzero(rng.random(n // 2) < 0.5) * 2:
            p[i], p[i + 1] = p[i + 1], p[i]
        rows = p[np.repeat(np.arange(n), np.diff(rp))]
        cols = p[ci]
        o = np.lexsort((cols, rows))
        rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
        ci, va = cols[o].astype(np.int32), va[o]
        c = np.empty_like(b)
        c[p] = b
        b = c
    B = ffhip.Matrix.upload(rp, ci, va)
    x, _ = ffhip.CG(B, layout="sell").solve(b, eps=1e-10)
    y, _ = ffhip.CG(B, layout="sell32").solve(b, eps=1e-10)
    assert np.linalg.norm(x - y) <= 1e-8 * np.linalg.norm(y)
