"""Which FP64 solves read half of the values (half_from: the first iteration that
does, 65 in a solver's first solve, 1 in the next, 0 where none does), and that
those that do give the whole matrix's solution bit for bit: the transposed solve
reads the whole matrix, and these matrices are symmetric.  Boxes, stencils of 4
to 6 neighbours before the diagonal, rows without a stored diagonal, and values
that lose their symmetry and regain it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")

BOX = (76, 77, 79)


def box_system():
    M = ffhip.cube(*BOX)
    A = ffhip.Matrix.p1(M)
    A.assemble_p1(ffhip.COEF_SIN3)
    labels = (1, 2, 3, 4, 5, 6)
    A.set_bc(labels)
    return A, ffhip.rhs_p1(M, 1.0, labels)


def solve(cg, b, **kw):
    x, st = cg.solve(b, eps=1e-6, itmax=300, raise_on_error=False, **kw)
    assert st["iters"] > 64 and np.isfinite(x).all()
    return x, st["half_from"]


def check(cg, b):
    """found in the first solve, used from the start in the second"""
    whole, none = solve(cg, b, trans=True)
    assert none == 0
    for first in (65, 1):
        x, half = solve(cg, b)
        assert half == first
        assert np.array_equal(x, whole)


@pytest.mark.parametrize("graph", [True, False])
def test_box(graph):
    A, b = box_system()
    check(ffhip.CG(A, graph=graph), b)


def stencil(nx, ny, offsets, holes=()):
    """symmetric matrix on an nx x ny grid: neighbours at +-(dx, dy), row sums
    positive; the rows in holes without a diagonal"""
    n = nx * ny
    i = np.arange(n)
    x, y = i % nx, i // nx
    rows, cols, vals = [], [], []
    diag = np.full(n, 0.01)
    for k, (dx, dy) in enumerate(offsets):
        ok = (x + dx >= 0) & (x + dx < nx) & (y + dy < ny)
        a, c = i[ok], i[ok] + dx + dy * nx
        v = -(1. + 0.1 * k + 0.05 * np.sin(0.01 * a))
        rows += [a, c]
        cols += [c, a]
        vals += [v, v]
        np.add.at(diag, a, -v)
        np.add.at(diag, c, -v)
    keep = np.setdiff1d(i, holes)
    rows, cols, vals = (np.concatenate(t) for t in (rows + [keep], cols + [keep], vals + [diag[keep]]))
    o = np.lexsort((cols, rows))
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    return rp, cols[o].astype(np.int32), vals[o]


NINE = [(1, 0), (-1, 1), (0, 1), (1, 1)]


@pytest.mark.parametrize("offsets", [NINE, NINE + [(0, 2)], NINE + [(0, 2), (2, 0)]], ids=["4", "5", "6"])
def test_stencils(offsets):
    rp, ci, va = stencil(1000, 900, offsets)
    b = np.random.default_rng(1).standard_normal(rp.size - 1)
    cg = ffhip.CG(ffhip.Matrix.upload(rp, ci, va))
    assert cg.layout()[0] == "sell16"
    check(cg, b)


def test_rows_without_a_diagonal():
    """a few rows inside, and the last one (its padding is no diagonal)"""
    nx, ny = 1000, 900
    rp, ci, va = stencil(nx, ny, NINE, holes=[0, 5 * nx + 7, 400 * nx + 500, nx * ny - 1])
    b = np.random.default_rng(2).standard_normal(nx * ny)
    cg = ffhip.CG(ffhip.Matrix.upload(rp, ci, va))
    out = []
    for trans in (True, False, False):
        x, st = cg.solve(b, eps=1e-14, itmax=150, raise_on_error=False, trans=trans)
        out.append((x, st["iters"]))
        assert st["half_from"] == (0, 65, 1)[len(out) - 1]
    for x, its in out[1:]:
        assert its == out[0][1] > 64 and np.array_equal(x, out[0][0])


def test_matrices_without_the_form():
    A, b = box_system()
    rp, ci, va = A.download()
    n = rp.size - 1
    rng = np.random.default_rng(1)
    p = np.arange(n)
    for i in np.flatnonzero(rng.random(n // 2) < 0.5) * 2:  # neighbours swapped at random
        p[i], p[i + 1] = p[i + 1], p[i]
    rows, cols = p[np.repeat(np.arange(n), np.diff(rp))], p[ci]
    o = np.lexsort((cols, rows))
    rq = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    c = np.empty_like(b)
    c[p] = b
    cg = ffhip.CG(ffhip.Matrix.upload(rq, cols[o].astype(np.int32), va[o]), layout="sell")
    for _ in range(2):
        assert solve(cg, c)[1] == 0


def test_new_values():
    """symmetric, one entry an ulp off its mirror, symmetric again"""
    A, b = box_system()
    rp, ci, va = A.download()
    rows = np.repeat(np.arange(rp.size - 1), np.diff(rp))
    off = va.copy()
    k = np.flatnonzero((ci < rows) & (va < 0))[1000]
    off[k] = np.nextafter(off[k], -1)
    B = ffhip.Matrix.upload(rp, ci, va)
    cg = ffhip.CG(B)
    check(cg, b)
    for _ in range(2):
        B.set_values(off)
        cg.update_values()
        for _ in range(2):
            assert solve(cg, b)[1] == 0
        B.set_values(va)
        cg.update_values()
        check(cg, b)
