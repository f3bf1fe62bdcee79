"""The work that a program of this library has it do, case by case, through its
public entry points: whole small scripts, matrix assembly with solver set-up,
re-assembly in a time loop, matrix products, the Krylov solves and the adjoint
blocks, in P1 (2D and 3D), scalar P2 and [P2,P2,P2].

A case is a dict: its `kind` picks the entry points, the rest are sizes and
options.  `prepare` makes what the program holds before the call (inputs from
the seed; for re-assembly, products and solves also the mesh, matrix or solver
it keeps), `run` is one pass and returns its outputs whole, `exact` computes
the same outputs with plain torch in 64 bits.
"""
import math
import os
import sys

import torch

sys.path.insert(1, os.path.join(os.getcwd(), "freefem-sources_amd"))
import ffhip  # noqa: E402

ALL = {2: (1, 2, 3, 4), 3: (1, 2, 3, 4, 5, 6)}
ROBIN, NEUMANN = (1, 2, 6), (3, 5)  # the heat step's boundary labels
CLAMPED = (4,)  # the elasticity cube hangs on its x = 0 face
COEF = {"const": ffhip.COEF_CONST, "sin3": ffhip.COEF_SIN3, "p0": ffhip.COEF_P0,
        "p1": ffhip.COEF_P1, "qp": ffhip.COEF_QP}
MODE = {"fp64": ffhip.CG_FP64, "mixed": ffhip.CG_MIXED}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # a whole script on a small ragged 2D mesh (mesh, matrix, Dirichlet
        # rows, right-hand side, solve): what a user's first script does, and
        # what an outer loop over small problems repeats; launches and waits
        dict(name="script2d_tiny", kind="script", nx=17, ny=13, nz=0, coef="p1", mode="fp64"),
        # the 2D Poisson configuration of the benchmark up to the solver
        dict(name="poisson2d_200", kind="poisson", nx=200, ny=200, nz=0, coef="p1", mode="fp64", bc=True),
        # the benchmark's main workload: cube(160), analytic kappa, mesh to
        # solver set-up; the largest assembly
        dict(name="poisson3d_160", kind="poisson", nx=160, ny=160, nz=160, coef="sin3", mode="fp64", bc=True),
        # one step of a time loop on a ragged box with a kept pattern:
        # stiffness, reaction and Robin terms, volume and Neumann right-hand sides
        dict(name="heat3d_odd", kind="heat", nx=61, ny=50, nz=43, coef="p0"),
        # the FP64 solve of the benchmark's main workload; the longest call
        dict(name="cg_fp64_160", kind="cg", nx=160, ny=160, nz=160, coef="sin3", mode="fp64"),
        # the FP32-inner / FP64-refinement solve at the middle 3D size
        dict(name="cg_mixed_64", kind="cg", nx=64, ny=64, nz=64, coef="sin3", mode="mixed"),
        # a non-symmetric system through solver=GMRES
        dict(name="gmres_20", kind="gmres", nx=20, ny=20, nz=20, coef="p0"),
        # matrix products of a script's own iteration: A*x, A'*x and the
        # product of the symmetric half-stored matrix (sym=1)
        dict(name="products_72", kind="products", nx=72, ny=72, nz=72, coef="p0"),
        # the benchmark's [P2,P2,P2] Lame cube, numbering to MIXED solver set-up
        dict(name="elasticity_32", kind="elasticity", nx=32, ny=32, nz=32, mode="mixed", bc=True),
        # its FP64 solve at a smaller size
        dict(name="elasticity_cg_20", kind="elasticity_cg", nx=20, ny=20, nz=20, mode="fp64"),
        # the scalar P2 Laplacian on a ragged box, numbering to solver set-up
        dict(name="p2_laplace_odd", kind="p2", nx=27, ny=24, nz=21, coef="p1", mode="fp64", bc=True),
        # the adjoint blocks of a coefficient inversion: misfit with its
        # adjoint right-hand side, then the element gradient
        dict(name="adjoint_96", kind="adjoint", nx=96, ny=96, nz=96),
    ]


# smallest and largest edge counts of the drawn boxes, per kind (2D, 3D)
RANGE = {"script": ((4, 120), (3, 36)), "poisson": ((8, 900), (6, 140)), "heat": (None, (6, 100)),
         "cg": (None, (10, 130)), "gmres": (None, (6, 26)), "products": (None, (8, 110)),
         "elasticity": (None, (3, 30)), "elasticity_cg": (None, (3, 20)), "p2": (None, (4, 40)),
         "adjoint": (None, (8, 120))}


def draw(rng):
    kind = rng.choice(sorted(RANGE))
    two = RANGE[kind][0] is not None and rng.random() < 0.5
    lo, hi = RANGE[kind][0 if two else 1]
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    dims = [max(2, min(hi, round(n * rng.uniform(0.8, 1.25)))) for _ in range(2 if two else 3)]
    case = dict(kind=kind, nx=dims[0], ny=dims[1], nz=0 if two else dims[2])
    if kind in ("script", "poisson", "heat", "cg", "gmres", "products", "p2"):
        case["coef"] = rng.choice(["p0", "p1"] if two else ["p0", "p1", "qp", "sin3"])
    if kind in ("script", "poisson", "cg", "elasticity", "elasticity_cg", "p2"):
        case["mode"] = rng.choice(["fp64", "mixed"])
    if kind in ("poisson", "elasticity", "p2"):
        case["bc"] = rng.random() < 0.5
    return case


# ---------------------------------------------------------------- sizes and inputs
def _dim(c):
    return 3 if c["nz"] else 2


def _sizes(c):
    """vertices, elements, boundary elements, edges"""
    x, y, z = c["nx"], c["ny"], c["nz"]
    if not z:
        return ((x + 1) * (y + 1), 2 * x * y, 2 * (x + y), x * (y + 1) + (x + 1) * y + x * y)
    edges = (x * (y + 1) * (z + 1) + (x + 1) * y * (z + 1) + (x + 1) * (y + 1) * z +
             x * y * (z + 1) + x * (y + 1) * z + (x + 1) * y * z + x * y * z)
    return (x + 1) * (y + 1) * (z + 1), 6 * x * y * z, 4 * (x * y + x * z + y * z), edges


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, dtype=torch.float64, device="cuda")


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, dtype=torch.float64, device="cuda")


def _coef_array(g, coef, c):
    """a lognormal coefficient of the kind's shape (None for the analytic ones)"""
    nv, nt = _sizes(c)[:2]
    if coef == "p0":
        return torch.exp(0.5 * _randn(g, nt))
    if coef == "p1":
        return torch.exp(0.5 * _randn(g, nv))
    if coef == "qp":
        return torch.exp(0.5 * _randn(g, nt, 14))
    return None


def _inputs(c, seed):
    g = _gen(seed)
    nv, nt, nbe = _sizes(c)[:3]
    d = {}
    if "coef" in c:
        d["kappa"] = _coef_array(g, c["coef"], c)
    k = c["kind"]
    if k in ("script", "poisson", "p2"):
        d["f"] = 0.5 + float(_rand(g, 1))
    elif k == "heat":
        d.update(mass=20. + 80. * _rand(g, nv), alpha=0.5 + _rand(g, nbe), f=_randn(g, nv), g=_randn(g, nbe))
    elif k in ("cg", "gmres"):  # a smooth source at the vertices
        X = _lattice(c) / torch.tensor([c["nx"], c["ny"], c["nz"]], dtype=torch.float64, device="cuda")
        a = _randn(g, 5)
        d["f"] = 1. + a[0] * torch.sin(3 * X[:, 0] + a[1]) + a[2] * torch.cos(4 * X[:, 1] + a[3]) * torch.sin(
            2 * X[:, 2] + a[4])
        if k == "gmres":
            d["skew"] = 0.5 * (1 + 0.1 * _randn(g, nv + 2 * _sizes(c)[3]))
    elif k == "products":
        d["skew"] = 0.5 * (1 + 0.1 * _randn(g, nv + 2 * _sizes(c)[3]))
        d["x"] = _randn(g, nv)
    elif k in ("elasticity", "elasticity_cg"):
        a = _rand(g, 5).tolist()
        d.update(lam=0.5 + a[0], mu=0.3 + a[1], fv=(a[2] - 0.5, a[3] - 0.5, a[4] - 1.5))
    elif k == "adjoint":
        d.update(u=_randn(g, nv), ud=_randn(g, nv), lam=_randn(g, nv))
    return d


# ---------------------------------------------------------------- the library's side
class _DeviceArray:
    """a device array of a matrix as torch takes it; holds the matrix's owners"""

    def __init__(self, ptr, n, typestr, owners):
        self.owners = owners
        self.__cuda_array_interface__ = dict(shape=(n,), typestr=typestr, data=(ptr, False), version=2)

    def tensor(self):
        return torch.as_tensor(self, device="cuda")


def _csr(A, *owners):
    rp, ci, va = A.device_ptrs()
    keep = (A,) + owners
    return dict(rowptr=_DeviceArray(rp, A.n + 1, "<i8", keep).tensor(),
                colidx=_DeviceArray(ci, A.nnz, "<i4", keep).tensor(),
                vals=_DeviceArray(va, A.nnz, "<f8", keep).tensor())


def _mesh(c):
    return ffhip.cube(c["nx"], c["ny"], c["nz"]) if c["nz"] else ffhip.square(c["nx"], c["ny"])


def _p1_matrix(c, mesh, kappa):
    if c["nz"]:
        return ffhip.Matrix.p1_assembled(mesh, COEF[c["coef"]], kappa_e=kappa)
    A = ffhip.Matrix.p1(mesh)
    A.assemble_p1(COEF[c["coef"]], kappa_e=kappa)
    return A


def _skew(A, w):
    """strictly upper entries scaled by w: a non-symmetric matrix on the same pattern"""
    m = _csr(A)
    rows = torch.repeat_interleave(torch.arange(A.n, device="cuda"), torch.diff(m["rowptr"]))
    m["vals"].mul_(torch.where(m["colidx"] > rows, w, torch.ones_like(w)))
    torch.cuda.synchronize()


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    k = c["kind"]
    s = dict(case=c, **d)
    if k == "heat":
        s["mesh"] = _mesh(c)
        s["A"] = ffhip.Matrix.p1(s["mesh"])
    elif k in ("cg", "gmres"):
        s["mesh"] = _mesh(c)
        s["A"] = _p1_matrix(c, s["mesh"], d["kappa"])
        if k == "gmres":
            _skew(s["A"], d["skew"])
        s["A"].set_bc(ALL[3])
        s["b"] = torch.empty(s["mesh"].nv, dtype=torch.float64, device="cuda")
        ffhip.rhs_p1_form(s["mesh"], ffhip.COEF_P1, fcoef=d["f"], labels=ALL[3], out=s["b"])
        s["cg"] = ffhip.CG(s["A"], MODE[c.get("mode", "fp64")])
    elif k == "products":
        s["mesh"] = _mesh(c)
        s["A"] = _p1_matrix(c, s["mesh"], d["kappa"])
        s["H"] = s["A"].lower()
        _skew(s["A"], d["skew"])
        for y in ("y", "yt", "yh"):
            s[y] = torch.empty_like(d["x"])
    elif k == "elasticity_cg":
        s["mesh"] = _mesh(c)
        s["space"] = ffhip.P2VSpace(s["mesh"])
        s["A"] = ffhip.Matrix.p2v(s["space"])
        s["A"].assemble_p2v_elasticity(d["lam"], d["mu"])
        s["A"].set_bc_p2v(CLAMPED)
        s["b"] = torch.empty(s["space"].ndof, dtype=torch.float64, device="cuda")
        ffhip.rhs_p2v(s["space"], d["fv"], CLAMPED, out=s["b"])
        s["cg"] = ffhip.CG(s["A"], MODE[c["mode"]])
    elif k == "adjoint":
        s["mesh"] = _mesh(c)
        # the incidence lists that the forward assembly leaves with the mesh
        ffhip.p1_misfit(s["mesh"], d["u"], d["ud"], ALL[3])
    return s


def run(s):
    c = s["case"]
    return globals()["_run_" + c["kind"]](s, c)


def _run_script(s, c):
    mesh = _mesh(c)
    labels = ALL[_dim(c)]
    A = _p1_matrix(c, mesh, s["kappa"])
    A.set_bc(labels)
    b = torch.empty(mesh.nv, dtype=torch.float64, device="cuda")
    ffhip.rhs_p1(mesh, s["f"], labels, out=b)
    u, _ = ffhip.CG(A, MODE[c["mode"]]).solve(b, eps=1e-10)
    return dict(u=u)


def _run_poisson(s, c):
    mesh = _mesh(c)
    labels = ALL[_dim(c)] if c["bc"] else ()
    A = _p1_matrix(c, mesh, s["kappa"])
    if c["bc"]:
        A.set_bc(labels)
    b = torch.empty(mesh.nv, dtype=torch.float64, device="cuda")
    ffhip.rhs_p1(mesh, s["f"], labels, out=b)
    cg = ffhip.CG(A, MODE[c["mode"]])
    return dict(_csr(A, mesh, cg), b=b)


def _run_heat(s, c):
    A, mesh = s["A"], s["mesh"]
    A.assemble_p1(COEF[c["coef"]], kappa_e=s["kappa"], mkind=ffhip.COEF_P1, mass_e=s["mass"])
    A.assemble_p1_boundary(ROBIN, ffhip.COEF_P0, coef=s["alpha"])
    b = torch.empty(mesh.nv, dtype=torch.float64, device="cuda")
    ffhip.rhs_p1_form(mesh, ffhip.COEF_P1, fcoef=s["f"], out=b)
    ffhip.rhs_p1_boundary(mesh, b, NEUMANN, ffhip.COEF_P0, coef=s["g"])
    return dict(vals=_csr(A, mesh)["vals"], b=b)


def _run_cg(s, c):
    x, _ = s["cg"].solve(s["b"], eps=1e-10)
    return dict(x=x)


def _run_gmres(s, c):
    x, _ = s["cg"].gmres(s["b"], eps=1e-10)
    return dict(x=x)


def _run_products(s, c):
    s["A"].spmv(s["x"], s["y"])
    s["A"].spmv(s["x"], s["yt"], trans=True)
    s["H"].spmv(s["x"], s["yh"])
    return dict(y=s["y"], yt=s["yt"], yh=s["yh"])


def _run_elasticity(s, c):
    mesh = _mesh(c)
    space = ffhip.P2VSpace(mesh)
    A = ffhip.Matrix.p2v(space)
    A.assemble_p2v_elasticity(s["lam"], s["mu"])
    labels = CLAMPED if c["bc"] else ()
    if c["bc"]:
        A.set_bc_p2v(labels)
    b = torch.empty(space.ndof, dtype=torch.float64, device="cuda")
    ffhip.rhs_p2v(space, s["fv"], labels, out=b)
    cg = ffhip.CG(A, MODE[c["mode"]])
    return dict(_csr(A, mesh, space, cg), b=b)


_run_elasticity_cg = _run_cg


def _run_p2(s, c):
    mesh = _mesh(c)
    space = ffhip.P2VSpace(mesh)
    A = ffhip.Matrix.p2(space)
    A.assemble_p2(COEF[c["coef"]], kappa_e=s["kappa"])
    labels = ALL[3] if c["bc"] else ()
    if c["bc"]:
        A.set_bc_p2(labels)
    b = torch.empty(space.nnodes, dtype=torch.float64, device="cuda")
    ffhip.rhs_p2(space, s["f"], labels, out=b)
    cg = ffhip.CG(A, MODE[c["mode"]])
    return dict(_csr(A, mesh, space, cg), b=b)


def _run_adjoint(s, c):
    J, r = ffhip.p1_misfit(s["mesh"], s["u"], s["ud"], ALL[3])
    g = ffhip.p1_grad_kappa(s["mesh"], s["u"], s["lam"])
    return dict(J=J, r=r, g=g)


# ---------------------------------------------------------------- work
def work(case):
    c, k, d = case, case["kind"], _dim(case)
    nv, nt, nbe, ne = _sizes(c)
    nnz, nodes = nv + 2 * ne, nv + ne
    mesh = 8 * d * nv + 4 * (d + 1) * nt + 4 * (d + 1) * nbe
    coef = {"p0": 8 * nt, "p1": 8 * nv, "qp": 112 * nt}.get(c.get("coef"), 0)
    side = max(c["nx"], c["ny"], c["nz"])
    p2nnz = 28 * nodes  # the P2 pattern: about 28 nodes a row on these meshes
    if k in ("script", "poisson"):
        out = dict(bytes=coef + mesh + 12 * nnz + 8 * nv + 8 * nv, flops=(900 if c["coef"] == "sin3" else 150) * nt)
        if k == "script":  # about 4 (2D: 2) iterations per edge count to 1e-10
            its = (4 if d == 3 else 2) * side
            out = dict(bytes=out["bytes"] + its * (12 * nnz + 92 * nv), flops=out["flops"] + its * (2 * nnz + 10 * nv))
        return out
    if k == "heat":
        return dict(bytes=coef + mesh + 8 * nv + 8 * nbe + 8 * nnz + 8 * nv + 8 * nbe + 8 * nv, flops=600 * nt)
    if k == "cg":
        its = 4 * side
        per = 12 * nnz + 92 * nv if c["mode"] == "fp64" else 8 * nnz + 48 * nv
        return dict(bytes=its * per, flops=its * (2 * nnz + 10 * nv))
    if k == "gmres":
        its = 3 * side
        return dict(bytes=its * (12 * nnz + 60 * nv) + 16 * its * its * nv, flops=its * 2 * nnz + 2 * its * its * nv)
    if k == "products":
        return dict(bytes=2 * (12 * nnz + 24 * nv) + 6 * nnz + 30 * nv, flops=6 * nnz)
    if k == "elasticity":
        return dict(bytes=mesh + 40 * nt + 108 * p2nnz + 48 * nodes, flops=28000 * nt)
    if k == "elasticity_cg":
        its = 50 * side + 200
        per = 76 * p2nnz + 276 * nodes if c["mode"] == "fp64" else 40 * p2nnz + 144 * nodes
        return dict(bytes=its * per, flops=its * 18 * p2nnz)
    if k == "p2":
        return dict(bytes=coef + mesh + 40 * nt + 12 * p2nnz + 16 * nodes, flops=26000 * nt)
    return dict(bytes=2 * mesh + 32 * nv + 8 * nv + 8 * nt, flops=250 * nt)


# ---------------------------------------------------------------- plain torch in 64 bits
_A, _B, _C = 0.31088591926330060980, 0.092735250310891226402, 0.045503704125649649492
_A0, _B0, _C0 = 1 - 3 * _A, 1 - 3 * _B, 0.5 - _C
TET5 = [(_B0, _B, _B), (_B, _B0, _B), (_B, _B, _B0), (_B, _B, _B), (_A0, _A, _A), (_A, _A0, _A), (_A, _A, _A0),
        (_A, _A, _A), (_C0, _C0, _C), (_C0, _C, _C0), (_C, _C0, _C0), (_C, _C, _C0), (_C, _C0, _C), (_C0, _C, _C)]
TET5_W = [0.073493043116361949544] * 4 + [0.11268792571801585080] * 4 + [0.042546020777081466438] * 6
SPLIT = [(4, 0, 6, 7), (0, 4, 5, 7), (1, 0, 5, 7), (0, 1, 3, 7), (2, 0, 3, 7), (0, 2, 6, 7)]
FACES = [(3, 2, 1), (0, 2, 3), (3, 1, 0), (0, 1, 2)]
EDGES = [(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)]


def _ar(n):
    return torch.arange(n, device="cuda")


def _lattice(c):
    k, j, i = torch.meshgrid(_ar(c["nz"] + 1), _ar(c["ny"] + 1), _ar(c["nx"] + 1), indexing="ij")
    return torch.stack([i, j, k], -1).reshape(-1, 3)


def _box(c):
    """vertices, elements, boundary elements, boundary labels of cube / square"""
    x, y, z = c["nx"], c["ny"], c["nz"]
    if not z:
        j, i = torch.meshgrid(_ar(y + 1), _ar(x + 1), indexing="ij")
        X = torch.stack([i.double() / x, j.double() / y], -1).reshape(-1, 2)
        i0 = (_ar(x) + (_ar(y) * (x + 1))[:, None]).reshape(-1)
        i1, i2, i3 = i0 + 1, i0 + x + 2, i0 + x + 1
        return X, torch.stack([i0, i1, i2, i0, i2, i3], -1).reshape(-1, 3), None, None
    idx = _lattice(c)
    X = idx.double() * torch.tensor([1. / x, 1. / y, 1. / z], dtype=torch.float64, device="cuda")
    nj, nk = x + 1, (x + 1) * (y + 1)
    base = (_ar(x) + nj * _ar(y)[:, None] + nk * _ar(z)[:, None, None]).reshape(-1)
    off = torch.tensor([a + nj * b + nk * e for e in (0, 1) for b in (0, 1) for a in (0, 1)], device="cuda")
    T = (base[:, None, None] + off[torch.tensor(SPLIT, device="cuda")][None]).reshape(-1, 4)
    bits = ((idx[:, 0] == 0) * 1 + (idx[:, 0] == x) * 2 + (idx[:, 1] == 0) * 4 + (idx[:, 1] == y) * 8 +
            (idx[:, 2] == 0) * 16 + (idx[:, 2] == z) * 32)
    f = T[:, torch.tensor(FACES, device="cuda")].reshape(-1, 3)
    m = bits[f[:, 0]] & bits[f[:, 1]] & bits[f[:, 2]]
    on = m != 0
    lab = torch.zeros(64, dtype=torch.int64, device="cuda")
    for bit, label in ((1, 4), (2, 2), (4, 1), (8, 3), (16, 5), (32, 6)):
        lab[bit] = label
    return X, T, f[on], lab[m[on]]


def _grads(X, T):
    """measures and P1 gradients of simplices"""
    d = X.shape[1]
    E = X[T[:, 1:]] - X[T[:, :1]]
    if d == 2:
        det = E[:, 0, 0] * E[:, 1, 1] - E[:, 0, 1] * E[:, 1, 0]
        N = torch.stack([torch.stack([E[:, 1, 1], -E[:, 1, 0]], -1), torch.stack([-E[:, 0, 1], E[:, 0, 0]], -1)], 1)
        vol = det / 2
    else:
        N = torch.stack([torch.linalg.cross(E[:, 1], E[:, 2]), torch.linalg.cross(E[:, 2], E[:, 0]),
                         torch.linalg.cross(E[:, 0], E[:, 1])], 1)
        det = (E[:, 0] * N[:, 0]).sum(-1)
        vol = det / 6
    G = N / det[:, None, None]
    return vol, torch.cat([-G.sum(1, keepdim=True), G], 1)


def _mean_coef(c, kappa, X, T):
    """the coefficient's mean over each element by the volume rule"""
    if c["coef"] == "p0":
        return kappa
    if c["coef"] == "p1":
        return kappa[T].mean(1)
    return sum(w * v for w, v in zip(TET5_W, _at_points(c, kappa, X, T)))


def _at_points(c, kappa, X, T):
    """the coefficient at the 14 points of every element"""
    for q, (a, b, e) in enumerate(TET5):
        lam = torch.tensor([1 - a - b - e, a, b, e], dtype=torch.float64, device="cuda")
        if c["coef"] == "p0":
            yield kappa
        elif c["coef"] == "p1":
            yield sum(lam[i] * kappa[T[:, i]] for i in range(4))
        elif c["coef"] == "qp":
            yield kappa.reshape(-1, 14)[:, q]
        else:
            s = 1.
            for axis in range(3):
                s = s * torch.sin(2 * math.pi * sum(lam[i] * X[T[:, i], axis] for i in range(4)))
            yield 1 + 0.5 * s


def _assemble(n, T, K):
    """CSR (rows, then columns, ascending) of element matrices K on dofs T"""
    m = T.shape[1]
    keys = (T[:, :, None] * n + T[:, None, :]).reshape(-1)
    keys, inv = torch.unique(keys, return_inverse=True)
    vals = torch.zeros(keys.numel(), dtype=torch.float64, device="cuda")
    vals.index_add_(0, inv, K.reshape(-1, m * m).reshape(-1))
    rows = torch.div(keys, n, rounding_mode="floor")
    rp = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    rp[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    return rp, (keys - rows * n).to(torch.int32), vals, rows


def _stiffness(c, kappa, X, T):
    vol, G = _grads(X, T)
    S = vol * _mean_coef(c, kappa, X, T)
    return S[:, None, None] * (G @ G.transpose(1, 2)), vol


def _load(n, T, vol, f):
    """int f v for P1 f (vertex values) or a constant"""
    m = T.shape[1]
    b = torch.zeros(n, dtype=torch.float64, device="cuda")
    if isinstance(f, float):
        e = (vol * f / m)[:, None].expand(-1, m)
    else:
        F = f[T]
        e = vol[:, None] * (F + F.sum(1, keepdim=True)) / (m * (m + 1))
    return b.index_add_(0, T.reshape(-1), e.reshape(-1))


def _boundary_dofs(c, n, X, labels=None):
    """the vertices (or P2 nodes) on the box's faces"""
    eps = 1e-9
    at = (X < eps) | (X > 1 - eps)
    return at.any(1) if labels is None else X[:, 0] < eps


def _p2_nodes(X, T):
    """P2 nodes by first appearance over (element, 4 vertices, 6 edges), and their points"""
    nv = X.shape[0]
    E = T[:, torch.tensor(EDGES, device="cuda")]
    key = torch.cat([T, nv + E.amin(-1) * nv + E.amax(-1)], 1).reshape(-1)
    u, inv = torch.unique(key, return_inverse=True)
    first = torch.full((u.numel(),), key.numel(), device="cuda").scatter_reduce_(0, inv, _ar(key.numel()), "amin")
    num = torch.empty_like(first)
    num[torch.argsort(first)] = _ar(u.numel())
    P = torch.cat([X[T], 0.5 * (X[E[:, :, 0]] + X[E[:, :, 1]])], 1).reshape(-1, 3)
    pts = torch.empty(u.numel(), 3, dtype=torch.float64, device="cuda")
    pts[num[inv]] = P
    return num[inv].reshape(-1, 10), pts


def _p2_gradients(G):
    """[element, basis, vertex v, axis]: gradients of the P2 basis as sums over v of l_v times these"""
    nt = G.shape[0]
    D = torch.zeros(nt, 10, 4, 3, dtype=torch.float64, device="cuda")
    for i in range(4):  # grad = G_i (4 l_i - 1), 1 = sum of the l_v
        D[:, i] -= G[:, i, None, :]
        D[:, i, i] += 4 * G[:, i]
    for e, (a, b) in enumerate(EDGES):
        D[:, 4 + e, a] += 4 * G[:, b]
        D[:, 4 + e, b] += 4 * G[:, a]
    return D


def _p2_load(n, N, vol, f):
    w = torch.tensor([-1 / 20] * 4 + [1 / 5] * 6, dtype=torch.float64, device="cuda")
    return torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(
        0, N.reshape(-1), (f * vol[:, None] * w).reshape(-1))


def _lame(X, T, lam, mu):
    """element matrices of the Lame form on dofs 3 node + component"""
    vol, G = _grads(X, T)
    D = _p2_gradients(G)
    m = (torch.ones(4, 4, dtype=torch.float64, device="cuda") + torch.eye(4, dtype=torch.float64, device="cuda")) / 20
    nt, out = T.shape[0], []
    for k in range(0, nt, 50000):
        d = D[k:k + 50000]
        # M[(i,a),(j,b)] = int d_a phi_i d_b phi_j
        left = d.permute(0, 1, 3, 2).reshape(-1, 30, 4)
        M = vol[k:k + 50000, None, None] * (left @ (left @ m).transpose(1, 2))
        M = M.reshape(-1, 10, 3, 10, 3)
        tr = M.diagonal(dim1=2, dim2=4).sum(-1)
        K = lam * M + mu * M.transpose(2, 4)
        for a in range(3):
            K[:, :, a, :, a] += mu * tr
        out.append(K.reshape(-1, 30, 30))
    return torch.cat(out), vol


def _krylov(rp, ci, va, b, fixed, symmetric=True, most=4000):
    """the solution with x = 0 on the fixed dofs: Jacobi CG (BiCGStab where the
    matrix is not symmetric), run until it no longer gains"""
    free = (~fixed).double()
    A = torch.sparse_csr_tensor(rp, ci.long(), va, (b.numel(), b.numel()))
    rows = torch.repeat_interleave(_ar(b.numel()), torch.diff(rp))
    diag = torch.zeros_like(b).index_add_(0, rows, torch.where(ci == rows, va, torch.zeros_like(va)))
    C = free / diag

    def mul(x):
        return free * (A @ (free * x))
    x, r = torch.zeros_like(b), free * b
    if symmetric:
        z = C * r
        p, rz = z.clone(), torch.dot(r, z)
        stop = 1e-31 * float(rz)
        for it in range(most):
            q = mul(p)
            a = rz / torch.dot(p, q)
            x += a * p
            r -= a * q
            z = C * r
            new = torch.dot(r, z)
            if it % 20 == 19 and float(new) < stop:
                break
            p = z + (new / rz) * p
            rz = new
        return x
    for _ in range(3):  # restarted on the true residual
        r = free * b - mul(x)
        r0, p = r.clone(), r.clone()
        rho = torch.dot(r0, r)
        stop = 1e-26 * float(rho)
        for it in range(most):
            if float(torch.dot(r, r)) <= max(stop, 1e-60):
                break
            y = C * p
            v = mul(y)
            a = rho / torch.dot(r0, v)
            s = r - a * v
            z = C * s
            t = mul(z)
            w = torch.dot(t, s) / torch.dot(t, t)
            x += a * y + w * z
            r = s - w * t
            new = torch.dot(r0, r)
            p = r + (new / rho) * (a / w) * (p - w * v)
            rho = new
    return x


def exact(case, seed):
    c, d, k = case, _inputs(case, seed), case["kind"]
    X, T, F, lab = _box(c)
    n = X.shape[0]
    if k == "adjoint":
        vol, G = _grads(X, T)
        e = (d["u"] - d["ud"])[T]
        J = (vol / 40 * ((e * e).sum(1) + e.sum(1) ** 2)).sum()
        r = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(
            0, T.reshape(-1), (vol[:, None] / 20 * (e + e.sum(1, keepdim=True))).reshape(-1))
        r[_boundary_dofs(c, n, X)] = 0.
        gu, gl = (torch.einsum("ei,eik->ek", v[T], G) for v in (d["u"], d["lam"]))
        return dict(J=float(J), r=r, g=-vol * (gu * gl).sum(1))
    if k in ("elasticity", "elasticity_cg", "p2"):
        N, P = _p2_nodes(X, T)
        nn = P.shape[0]
        if k == "p2":
            vol, G = _grads(X, T)
            D = _p2_gradients(G)
            K = torch.zeros(T.shape[0], 10, 10, dtype=torch.float64, device="cuda")
            for (a, b, e), w, kq in zip(TET5, TET5_W, _at_points(c, d["kappa"], X, T)):
                lam = torch.tensor([1 - a - b - e, a, b, e], dtype=torch.float64, device="cuda")
                g = torch.einsum("eivk,v->eik", D, lam)
                K += (vol * w * kq)[:, None, None] * (g @ g.transpose(1, 2))
            fixed = _boundary_dofs(c, nn, P) if c["bc"] else torch.zeros(nn, dtype=torch.bool, device="cuda")
            b = _p2_load(nn, N, vol, d["f"])
        else:
            K, vol = _lame(X, T, d["lam"], d["mu"])
            clamp = _boundary_dofs(c, nn, P, CLAMPED) & bool(c.get("bc", True))
            fixed = clamp.repeat_interleave(3)
            b = torch.stack([_p2_load(nn, N, vol, f) for f in d["fv"]], 1).reshape(-1)
            N = (3 * N[:, :, None] + _ar(3)).reshape(-1, 30)
            nn *= 3
        rp, ci, va, rows = _assemble(nn, N, K)
    else:
        K, vol = _stiffness(c, d["kappa"], X, T)
        nn = n
        fixed = _boundary_dofs(c, n, X) if c.get("bc", k in ("script", "cg", "gmres")) else torch.zeros(
            n, dtype=torch.bool, device="cuda")
        if k == "heat":  # int m u v with P1 m: int l_a l_i l_j over a simplex by the factorial rule
            m3 = torch.empty(4, 4, 4, dtype=torch.float64, device="cuda")
            for a in range(4):
                for i in range(4):
                    for j in range(4):
                        m3[a, i, j] = math.prod(math.factorial([a, i, j].count(t)) for t in range(4)) * 6 / 720
            K += vol[:, None, None] * torch.einsum("ea,aij->eij", d["mass"][T], m3)
        rp, ci, va, rows = _assemble(n, T, K)
        b = None if k == "products" else _load(n, T, vol, d["f"])
    del K
    if k == "heat":
        area = 0.5 * torch.linalg.cross(X[F[:, 1]] - X[F[:, 0]], X[F[:, 2]] - X[F[:, 0]]).norm(dim=1)

        def on(labels):
            return sum((lab == q) for q in labels).double()
        w = on(ROBIN) * d["alpha"] * area / 12
        M = w[:, None, None] * (1 + torch.eye(3, dtype=torch.float64, device="cuda"))
        keys = rows * n + ci
        at = torch.searchsorted(keys, (F[:, :, None] * n + F[:, None, :]).reshape(-1))
        va.index_add_(0, at, M.reshape(-1))
        b.index_add_(0, F.reshape(-1), (on(NEUMANN) * d["g"] * area / 3)[:, None].expand(-1, 3).reshape(-1))
        return dict(vals=va, b=b)
    if k in ("gmres", "products"):
        sym = va.clone()
        va = va * torch.where(ci > rows, d["skew"], torch.ones_like(va))
    if k == "products":
        x = d["x"]

        def mul(v, r, q):
            return torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, r, v * x[q])
        ci = ci.long()
        return dict(y=mul(va, rows, ci), yt=mul(va, ci, rows), yh=mul(sym, rows, ci))
    if k in ("poisson", "elasticity", "p2"):
        va[(ci == rows) & fixed[rows]] = 1e30
        b[fixed] = 0.
        return dict(rowptr=rp, colidx=ci, vals=va, b=b)
    x = _krylov(rp, ci, va, b, fixed, symmetric=k != "gmres")
    return dict(u=x) if k == "script" else dict(x=x)
