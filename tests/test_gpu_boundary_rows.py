"""Boundary integrals at the edges of a wave's 16 vertices and 64 items: vertex
counts off 16, waves that hold a plane of boundary vertices (more than 64 items)
or none, a vertex of 80 boundary triangles, some labels only; matrix and
right-hand side against the oracle.  Bars as in the boundary tests."""
import numpy as np
import pytest

import ffo
from test_gpu_p1 import _fan_mesh, _vals_close

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")

MESHES = {"box111": lambda: ffo.cube(1, 1, 1), "box15": lambda: ffo.cube(15, 1, 1), "box20": lambda: ffo.cube(20, 9, 3),
          "box12": lambda: ffo.cube(12, 11, 13), "fan": lambda: _fan_mesh(80), "square": lambda: ffo.square(37, 21)}


@pytest.mark.parametrize("name", MESHES)
def test_boundary_rows(name):
    mo = MESHES[name]()
    two = name == "square"
    nloc, el, be = (3, mo["tris"], mo["bedges"]) if two else (4, mo["tets"], mo["btri"])
    dim = 2 if two else 3
    labels, dirichlet = ((1, 3), (2,)) if name != "fan" else ((1,), ())
    m = (ffhip.mesh2_upload(mo["xy"], el, be, mo["blab"]) if two
         else ffhip.mesh3_upload(mo["xyz"], el, be, mo["blab"]))
    rp, ci = ffo.pattern(mo["nv"], el, nloc)
    vo = (ffo.assemble_p1_2d if two else ffo.assemble_p1_3d)(mo, rp, ci, ffo.COEF_SIN3)
    ce = np.random.default_rng(3).uniform(0.5, 2.0, mo["nbe"])
    ffo.p1_boundary(mo, labels, ffo.COEF_P0, 0.0, coef=ce, rowptr=rp, colidx=ci, vals=vo)
    A = ffhip.Matrix.p1(m)
    A.assemble_p1(ffhip.COEF_SIN3)
    A.assemble_p1_boundary(labels, ffhip.COEF_P0, 0.0, ce)
    assert _vals_close(A.download()[2], vo)
    bo = (ffo.rhs_p1_2d if two else ffo.rhs_p1_3d)(mo, 1.0)
    ffo.p1_boundary(mo, labels, ffo.COEF_SIN3, 0.0, b=bo)
    b = ffhip.rhs_p1(m, 1.0, dirichlet, 1e30, 0.25)
    if dirichlet:
        ffo.rhs_bc(bo, ffo.mark_bc(mo["nv"], be, mo["blab"], dim, dirichlet), 1e30, 0.25)
    ffhip.rhs_p1_boundary(m, b, labels, ffhip.COEF_SIN3, 0.0, dirichlet=dirichlet)
    big = bo >= 1e29
    assert np.array_equal(b[big], bo[big])
    assert np.abs(b - bo)[~big].max(initial=0) <= 1e-12 * np.abs(bo[~big]).max(initial=1e-300)
