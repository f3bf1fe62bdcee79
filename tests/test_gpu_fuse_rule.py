"""Which systems form the CG direction in the mat-vec: it gathers two vectors per
entry, which pays where consecutive rows hold consecutive columns (box meshes)
or the system is small, and costs up to twice the time in an arbitrary
numbering.  Both ways solve the same system: the renumbered mesh's solution is
the box's (bar of the CG tests: 1e-8)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


def renumbered(n, within=None):
    d = ffhip.cube(n).download()
    place = np.arange(d["nv"]) + np.random.default_rng(n).uniform(0, within or 10 * d["nv"], d["nv"])
    p = np.empty(d["nv"], np.int32)
    p[np.argsort(place)] = np.arange(d["nv"])
    xyz = np.empty((d["nv"], 3))
    xyz[p] = d["xyz"].reshape(-1, 3)
    return ffhip.mesh3_upload(xyz, p[d["elems"]], p[d["belems"]], d["blab"]), p


def solve(A, b, mode, layout="auto"):
    x, st = ffhip.CG(A, mode, layout).solve(b, eps=1e-10)
    assert st["converged"] == 1
    return x, st["fused"]


def system(M):
    A = ffhip.Matrix.p1(M)
    A.assemble_p1(ffhip.COEF_SIN3)
    labels = (1, 2, 3, 4, 5, 6)
    A.set_bc(labels)
    return A, ffhip.rhs_p1(M, 1.0, labels)


# rows: 2744, 12167 (small in both), 17576 (FP64 needs the order), 35937 (both do)
@pytest.mark.parametrize("n,box,random", [(13, (0, 1), (0, 1)), (22, (1, 1), (1, 1)), (25, (1, 1), (0, 1)),
                                          (32, (1, 1), (0, 0))])
def test_rule(n, box, random):
    A, b = system(ffhip.cube(n))
    M, p = renumbered(n)
    B, c = system(M)
    for mode in (ffhip.CG_FP64, ffhip.CG_MIXED):
        x, fx = solve(A, b, mode)
        y, fy = solve(B, c, mode)
        assert (fx, fy) == (box[mode], random[mode])
        assert np.linalg.norm(y[p] - x) <= 1e-8 * np.linalg.norm(x)


@pytest.mark.parametrize("mesh", [lambda: ffhip.square(255), lambda: ffhip.square(511), lambda: ffhip.cube(63),
                                  lambda: ffhip.cube(31, 63, 63), lambda: ffhip.cube(15, 127, 63)])
def test_lines_of_a_power_of_two(mesh):
    """65536 to 262144 rows: an even spread of samples would meet the lines' ends"""
    M = mesh()
    A = ffhip.Matrix.p1(M)
    A.assemble_p1(ffhip.COEF_CONST, 1.0)
    A.set_bc((1, 2, 3))
    b = ffhip.rhs_p1(M, 1.0, (1, 2, 3))
    for mode in (ffhip.CG_FP64, ffhip.CG_MIXED):
        assert solve(A, b, mode)[1] == 1


# 68921 and 262144 rows in FP64 and MIXED (2^18 is the limit), 274625 past it
@pytest.mark.parametrize("n,fused", [(40, 1), (63, 1), (64, 0)])
def test_shuffled_within_a_few(n, fused):
    A, b = system(renumbered(n, 30)[0])
    for mode in (ffhip.CG_FP64, ffhip.CG_MIXED):
        assert solve(A, b, mode)[1] == fused


def test_other_layouts():
    A, b = system(ffhip.cube(32))
    for layout in ("csr", "sell32"):
        for mode in (ffhip.CG_FP64, ffhip.CG_MIXED):
            assert solve(A, b, mode, layout)[1] == 0
    S = ffhip.P2VSpace(ffhip.cube(16))  # 35937 nodes, numbered by first appearance
    A = ffhip.Matrix.p2(S)
    A.assemble_p2()
    A.set_bc_p2((1, 2, 3, 4, 5, 6))
    for mode in (ffhip.CG_FP64, ffhip.CG_MIXED):
        assert solve(A, ffhip.rhs_p2(S, 1.0, (1, 2, 3, 4, 5, 6)), mode)[1] == 0
