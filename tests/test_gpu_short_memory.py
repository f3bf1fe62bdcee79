"""Calls on a device whose memory has run out.  hipMalloc and hipHostMalloc as
libffhip calls them go through Python here (their slots in the library's table
of imported functions), which fails the chosen requests by asking the runtime
for 2^60 bytes: the error, and the last error it leaves, are the runtime's own."""
import ctypes
import struct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ffhip = pytest.importorskip("ffhip")
ERR_HIP = -2


def import_slots(path):
    """offset of each imported function's slot from the library's load address"""
    f = open(path, "rb").read()
    shoff, = struct.unpack_from("<Q", f, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", f, 0x3A)
    sections = [struct.unpack_from("<IIQQQQIIQQ", f, shoff + i * shentsize) for i in range(shnum)]
    slots = {}
    for _, kind, _, _, off, size, link, _, _, _ in sections:
        if kind != 4:  # SHT_RELA
            continue
        symoff, strlink = sections[link][4], sections[link][6]
        stroff = sections[strlink][4] if strlink else 0
        for o in range(off, off + size, 24):
            where, info, _ = struct.unpack_from("<QQq", f, o)
            if info & 0xffffffff == 7:  # R_X86_64_JUMP_SLOT
                name, = struct.unpack_from("<I", f, symoff + 24 * (info >> 32))
                slots[f[stroff + name:f.index(b"\0", stroff + name)].decode()] = where
    return slots


class Allocator:
    def __init__(self):
        L = ffhip.lib()
        ffhip.context()
        path = ffhip.LIBPATH
        base = min(int(l.split("-")[0], 16) for l in open("/proc/self/maps") if l.rstrip().endswith(path))
        slots = import_slots(path)
        self.fail = lambda size: False
        self.fail_host = lambda size: False
        self.kept = []
        for name, sig, rule in (("hipMalloc", ctypes.c_size_t, "fail"),
                                ("hipHostMalloc", ctypes.c_size_t, "fail_host")):
            real = getattr(L, name)
            extra = [ctypes.c_uint] if name == "hipHostMalloc" else []
            real.argtypes = [ctypes.c_void_p, sig] + extra
            real.restype = ctypes.c_int
            proto = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, sig, *extra)

            def call(p, size, *flags, real=real, rule=rule):
                return real(p, (1 << 60) if getattr(self, rule)(size) else size, *flags)
            slot = ctypes.c_void_p.from_address(base + slots[name])
            self.kept.append((slot, slot.value, proto(call)))
            slot.value = ctypes.cast(self.kept[-1][2], ctypes.c_void_p).value

    def drop_cache(self):
        """the library gives its cached blocks back when a request fails"""
        self.fail = lambda size: True
        with pytest.raises(ffhip.FFHipError) as e:
            ffhip.cube(390, 380, 400)  # 5.7 GB of tets: larger than any block kept
        assert e.value.code == ERR_HIP
        self.fail = lambda size: False

    def limit(self, size, count):
        """requests for a block of `size` bytes fail after `count` of them"""
        left = [count]

        def fail(s):
            if size <= s < size + 256:
                left[0] -= 1
            return left[0] < 0 and size <= s < size + 256
        self.fail = fail

    def close(self):
        for slot, old, _ in self.kept:
            slot.value = old


@pytest.fixture
def alloc():
    a = Allocator()
    yield a
    a.close()


def rotation(n):
    rng = np.random.default_rng(n)
    i = np.arange(n)
    M = np.zeros((n, n))
    M[i, i] = 1.5 + 0.05 * rng.standard_normal(n)
    M[i[:-1], i[:-1] + 1] = 1.0
    M[i[1:], i[1:] - 1] = -0.9
    rows, ci = np.nonzero(M)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    return ffhip.Matrix.upload(rp, ci.astype(np.int32), M[rows, ci]), rng.standard_normal(n)


def test_gmres_takes_the_vectors_that_fit(alloc):
    n = 3000
    A, b = rotation(n)
    x0, s0 = ffhip.CG(A).gmres(b, eps=1e-10)
    its = s0["iters"]
    assert s0["converged"] == 1 and its > 12
    for pairs in (its + 1, its + 3, 5):
        cg = ffhip.CG(A)
        alloc.drop_cache()
        alloc.limit(8 * n, 2 + 2 * pairs + 1)  # w and x0, the pairs, and half of one more
        if pairs > its:  # a batch cut short, the same arithmetic
            x, st = cg.gmres(b, eps=1e-10)
            assert st["iters"] == its and np.array_equal(x, x0)
        else:
            with pytest.raises(ffhip.FFHipError) as e:
                cg.gmres(b, eps=1e-10)
            assert e.value.code == ERR_HIP
            alloc.fail = lambda size: False
            x, st = cg.gmres(b, eps=1e-10)  # room again
            assert st["iters"] == its and np.array_equal(x, x0)
        alloc.fail = lambda size: False


def test_gmres_after_a_failed_page_locked_buffer(alloc):
    n = 3000
    A, b = rotation(n)
    x0, _ = ffhip.CG(A).gmres(b, eps=1e-10)
    cg = ffhip.CG(A)
    alloc.fail_host = lambda size: True
    with pytest.raises(ffhip.FFHipError) as e:
        cg.gmres(b, eps=1e-10)
    assert e.value.code == ERR_HIP
    alloc.fail_host = lambda size: False
    assert np.array_equal(cg.gmres(b, eps=1e-10)[0], x0)


@pytest.mark.parametrize("labels", [(), (1, 3, 5), tuple(range(3, 40))])
def test_misfit_without_room_for_the_element_pairs(alloc, labels):
    import torch
    M = ffhip.cube(13, 11, 9)
    g = torch.Generator().manual_seed(3)
    u, ud = (torch.randn(M.nv, generator=g, dtype=torch.float64).cuda() for _ in range(2))
    J0, r0 = ffhip.p1_misfit(M, u, ud, labels)
    alloc.drop_cache()
    alloc.limit(16 * M.nt, 0)
    J, r = ffhip.p1_misfit(M, u, ud, labels)
    assert J == J0 and torch.equal(r, r0)


@pytest.mark.parametrize("kind,entries,size", [(ffhip.COEF_CONST, 0, 1), (ffhip.COEF_P0, 1, 1), (ffhip.COEF_P1, -1, 2),
                                               (ffhip.COEF_SIN3, 0, 4), (ffhip.COEF_QP, 14, 4)])
@pytest.mark.parametrize("labels", [(), (2, 5)])
def test_rhs_without_room_for_every_tet(alloc, kind, entries, size, labels):
    import torch
    M = ffhip.cube(13, 11, 9)  # 7722 tets
    g = torch.Generator().manual_seed(4)
    f = torch.randn(M.nv if entries < 0 else entries * M.nt, generator=g, dtype=torch.float64).cuda() if entries else None
    gv = torch.randn(M.nv, generator=g, dtype=torch.float64).cuda()
    b0, b = (torch.full((M.nv,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(2))
    ffhip.rhs_p1_form(M, kind, 1.5, f, labels, gvals=gv, out=b0)
    alloc.drop_cache()
    for parts in (1, 3):  # halves, then eighths
        sizes = [8 * size * (-(-M.nt // 2 ** k)) for k in range(parts)]
        alloc.fail = lambda s: any(q <= s < q + 256 for q in sizes)
        ffhip.rhs_p1_form(M, kind, 1.5, f, labels, gvals=gv, out=b)
        assert torch.equal(b, b0)
        b.fill_(float("nan"))
        alloc.drop_cache()


def test_half_of_the_values_without_room(alloc):
    M = ffhip.cube(76, 77, 79)
    A = ffhip.Matrix.p1(M)
    A.assemble_p1(ffhip.COEF_SIN3)
    A.set_bc((1, 2, 3, 4, 5, 6))
    b = ffhip.rhs_p1(M, 1.0, (1, 2, 3, 4, 5, 6))
    cg = ffhip.CG(A)
    x0, st = cg.solve(b, eps=1e-6, trans=True)
    assert st["iters"] > 64
    alloc.drop_cache()
    half = -(-M.nv // 64) * 64 * 8 * 8  # 8 values a row, rounded to 2 MiB by the allocator
    alloc.fail = lambda size: half <= size <= half + (2 << 20)
    for _ in range(2):
        x, st = cg.solve(b, eps=1e-6)
        assert st["half_from"] == 0 and np.array_equal(x, x0)
    alloc.fail = lambda size: False
    cg.update_values()  # looked for again
    x, st = cg.solve(b, eps=1e-6)
    assert st["half_from"] == 65 and np.array_equal(x, x0)
