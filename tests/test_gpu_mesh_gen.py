"""Device-built cube and square meshes, array by array against the oracle's
BuildCube / Carre_ restatements: single hexes, thin boxes in every direction,
sizes around the 256 hexes of a block."""
import numpy as np
import pytest

import ffo

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")


@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 1), (1, 2, 1), (1, 1, 2), (1, 5, 7), (6, 1, 9), (8, 4, 1),
                                  (255, 1, 1), (1, 257, 1), (1, 1, 256), (16, 16, 1), (7, 37, 2), (13, 11, 9)])
def test_cube(dims):
    lab = (4, 9, 2, 7, 1, 3)
    m, o = ffhip.cube(*dims, labels=lab).download(), ffo.cube(*dims, labels=lab)
    assert (m["nv"], m["nt"], m["nbe"]) == (o["nv"], o["nt"], o["nbe"])
    for a, b in (("xyz", "xyz"), ("elems", "tets"), ("belems", "btri"), ("blab", "blab")):
        assert np.array_equal(m[a], o[b]), a


@pytest.mark.parametrize("dims", [(1, 1), (1, 300), (257, 1), (3, 2), (31, 17)])
def test_square(dims):
    lab = (4, 9, 2, 7)
    m, o = ffhip.square(*dims, labels=lab).download(), ffo.square(*dims, labels=lab)
    assert (m["nv"], m["nt"], m["nbe"]) == (o["nv"], o["nt"], o["nbe"])
    for a, b in (("xyz", "xy"), ("elems", "tris"), ("belems", "bedges"), ("blab", "blab")):
        assert np.array_equal(m[a], o[b]), a
