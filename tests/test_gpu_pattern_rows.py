"""P1 rows of 1 to 40 elements (32 is the half-wave's limit), of 32, 33, 64 and
more columns, with vertex ids that collide in the row's set of columns: fans of
tetrahedra around an edge and stars of tetrahedra that share one vertex, their
vertices renumbered at random; fans of triangles in 2D.  Bars as in the P1
tests: patterns bit-exact, values within 1e-12 of the largest entry, the
one-call assembly equal to the two calls bit for bit."""
import numpy as np
import pytest

import ffo

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


def fans(sizes, stars, seed):
    rng = np.random.default_rng(seed)
    X, T = [], []
    for k in sizes:  # k tets around the edge (o, o + 1), a closed ring
        o = len(X)
        X += [[0, 0, -1], [0, 0, 1]] + [[np.cos(t), np.sin(t), 0.1 * np.cos(3 * t)]
                                         for t in 2 * np.pi * np.arange(k) / k]
        T += [[o, o + 1, o + 2 + i, o + 2 + (i + 1) % k] for i in range(k)]
    for k in stars:  # k tets that share only o
        o = len(X)
        X.append([0, 0, 0])
        for i in range(k):
            b = len(X)
            X += (np.eye(3) + 0.2 * rng.random((3, 3))).tolist()
            T.append([o, b, b + 1, b + 2])
    X, T = np.array(X, float), np.array(T, np.int32)
    p = rng.permutation(len(X)).astype(np.int32)
    Y = np.empty_like(X)
    Y[p] = X
    T = p[T]
    for t in T:  # each tet's own vertex order, positive volume
        t[:] = rng.permutation(t)
        A = Y[t[1:]] - Y[t[0]]
        if np.linalg.det(A) < 0:
            t[[1, 2]] = t[[2, 1]]
    T = T[rng.permutation(len(T))]
    return dict(nv=len(X), nt=len(T), nbe=0, xyz=Y.ravel().copy(), tets=T.ravel().copy(),
                btri=np.zeros(0, np.int32), blab=np.zeros(0, np.int32))


@pytest.mark.parametrize("sizes,stars", [((3, 4, 31, 32), (1,)), ((33, 40), (2,)), (tuple(range(3, 35)), (10,)),
                                         ((5,), (20, 21, 22, 32, 33)), ((6,) * 400, (7,) * 100)])
def test_rows_3d(sizes, stars):
    mo = fans(sizes, stars, len(sizes))
    rp, ci = ffo.pattern(mo["nv"], mo["tets"], 4)
    ke = np.exp(0.5 * np.random.default_rng(1).standard_normal(mo["nt"]))
    vo = ffo.assemble_p1_3d(mo, rp, ci, ffo.COEF_P0, 1.0, ke)
    m = ffhip.mesh3_upload(mo["xyz"], mo["tets"], mo["btri"], mo["blab"])
    one = ffhip.Matrix.p1_assembled(m, ffhip.COEF_P0, 1.0, ke)
    two = ffhip.Matrix.p1(ffhip.mesh3_upload(mo["xyz"], mo["tets"], mo["btri"], mo["blab"]))
    two.assemble_p1(ffhip.COEF_P0, 1.0, ke)
    a, b = one.download(), two.download()
    assert np.array_equal(a[0], rp) and np.array_equal(a[1], ci)
    assert np.abs(a[2] - vo).max() <= 1e-12 * np.abs(vo).max()
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("sizes", [(1, 2, 3), (31, 32, 33, 40), tuple(range(3, 35))])
def test_rows_2d(sizes):
    rng = np.random.default_rng(2)
    X, T = [], []
    for k in sizes:  # k triangles around o, open
        o = len(X)
        X += [[0, 0]] + [[np.cos(t), np.sin(t)] for t in 6 * np.arange(k + 1) / (k + 1)]
        T += [[o, o + 1 + i, o + 2 + i] for i in range(k)]
    X, T = np.array(X, float), np.array(T, np.int32)
    p = rng.permutation(len(X)).astype(np.int32)
    Y = np.empty_like(X)
    Y[p] = X
    T = np.array([np.roll(t, rng.integers(3)) for t in p[T]], np.int32)
    mo = dict(nv=len(X), nt=len(T), nbe=0, xy=Y.ravel().copy(), tris=T.ravel().copy(),
              bedges=np.zeros(0, np.int32), blab=np.zeros(0, np.int32))
    rp, ci = ffo.pattern(mo["nv"], mo["tris"], 3)
    vo = ffo.assemble_p1_2d(mo, rp, ci, ffo.COEF_CONST)
    A = ffhip.Matrix.p1(ffhip.mesh2_upload(mo["xy"], mo["tris"], mo["bedges"], mo["blab"]))
    A.assemble_p1(ffhip.COEF_CONST)
    rpa, cia, va = A.download()
    assert np.array_equal(rpa, rp) and np.array_equal(cia, ci)
    assert np.abs(va - vo).max() <= 1e-12 * np.abs(vo).max()
