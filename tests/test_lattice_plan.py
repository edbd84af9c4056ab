"""The split of a box into workgroups (lattice_plan of lattice.hip), on the host:
every cell and every node after a tile has its thread, whatever the box.  CPU only."""
import ctypes as C

import pytest

from fempar_amd import _native as N


class Lattice(C.Structure):
    _fields_ = [("nc", C.c_int * 3), ("m", C.c_int * 3), ("o", C.c_int * 3), ("E", C.c_int * 3), ("TX", C.c_int),
                ("TY", C.c_int), ("xt", C.c_int), ("tiles", C.c_int), ("nch", C.c_int), ("stride", C.c_int)]


class LatticeOp(C.Structure):
    _fields_ = [("g", Lattice), ("dim", C.c_int), ("order", C.c_int), ("ncomp", C.c_int), ("one", C.c_bool),
                ("threads", C.c_int), ("grid", C.c_int), ("lds", C.c_size_t), ("identity", C.c_bool),
                ("rounds", C.c_int), ("layers", C.c_int)]


def plan(n, order, ncomp, bc, cus=256, max_threads=0, cells=0):
    f = C.CDLL(N.LIB_PATH)._ZN6femhip12lattice_planERK18femhip_mesh_desc_tiRNS_9LatticeOpEii
    f.restype = C.c_bool
    f.argtypes = [C.POINTER(N.MeshDesc), C.c_int, C.POINTER(LatticeOp), C.c_int, C.c_int]
    d = N.MeshDesc(dim=len(n), order=order, num_components=ncomp, dirichlet=bc)
    for k in range(3):
        d.n[k] = n[k] if k < len(n) else 1
        d.limits[2 * k + 1] = 1.0
    L = LatticeOp()
    return L if f(C.byref(d), cus, C.byref(L), max_threads, cells) else None


def check_tiles(L, most):
    g, p = L.g, L.order
    E = [g.E[0], g.E[1] if L.dim == 3 else 1]
    yt = g.tiles // g.xt
    assert g.tiles == g.xt * yt and g.xt >= 1 and yt >= 1
    for e, t, count in ((E[0], g.TX, g.xt), (E[1], g.TY, yt)):   # neighbours share a row of cells
        assert t >= min(e, 2) and count * (t - 1) + 1 >= e
    halo = p * (g.TX + g.TY) + 1 if L.dim == 3 else 1            # nodes after the tile, one a thread
    assert max(g.TX * g.TY, halo) <= L.threads <= most
    assert L.lds <= 160 * 1024
    assert 1 <= g.nch <= g.E[L.dim - 1] and L.grid >= g.tiles * g.nch


@pytest.mark.parametrize("order,ncomp", [(1, 1), (1, 3), (2, 1)])
@pytest.mark.parametrize("bc", [N.BC_ALL_BOUNDARY, N.BC_X0_FACE, N.BC_NONE])
def test_tiles_cover_thin_boxes(order, ncomp, bc):
    """One to four cells along x, every length along y up to 800; a few lengths
    along z take both forms of an iteration.  A Q1 box with no free node is refused."""
    most = {(1, 1): 768, (1, 3): 512, (2, 1): 256}[order, ncomp]
    for nx in (1, 2, 3, 4):
        for ny in range(1, 801):
            for nz in (5, 2000):
                L = plan((nx, ny, nz), order, ncomp, bc)
                if bc == N.BC_ALL_BOUNDARY and order == 1 and min(nx, ny) < 2:
                    assert L is None
                else:
                    assert L, (nx, ny, nz)
                    check_tiles(L, most)


@pytest.mark.parametrize("order", [1, 2])
def test_tiles_cover_boxes(order):
    for nx, ny in ((5, 700), (63, 9), (64, 64), (127, 2), (128, 3), (255, 2), (256, 2), (1000, 2), (2000, 5), (3, 3000)):
        for bc in (N.BC_ALL_BOUNDARY, N.BC_X0_FACE, N.BC_NONE):
            L = plan((nx, ny, 7), order, 1, bc)
            assert L, (nx, ny)
            check_tiles(L, 768 if order == 1 else 256)
            L = plan((nx, ny), order, 1, bc)
            assert L
            check_tiles(L, 768)


def window_rows(L, chunk):
    """lattice_window of lattice.h: rows of the whole planes that a chunk of the march reads."""
    g, a, p = L.g, L.dim - 1, L.order
    z0, z1 = g.E[a] * chunk // g.nch, g.E[a] * (chunk + 1) // g.nch
    first, last = max(p * max(z0 - 1, 0) - g.o[a], 0), min(p * z1 - g.o[a], g.m[a] - 1)
    return max(last - first + 1, 0) * (g.m[0] * g.m[1] if L.dim == 3 else g.m[0])


@pytest.mark.parametrize("dim,sizes", [
    (2, (130, 1000, 2048, 4095, 4096)),
    (3, (25, 100, 400, 512, 513, 514, 515, 600, 647, 813, 814, 1000, 1030, 1290, 1291))])
def test_batch_windows_keep_their_byte_offsets(dim, sizes):
    """The passes of a batch read vectors of any length through windows of at
    most 2^30 bytes: larger ones would reach the offsets that stand for `outside'.
    Cells a workgroup as plan_passes asks for them."""
    for n in sizes:
        rows = (n - 1) ** dim
        for per in (1024, 16384):
            L = plan((n,) * dim, 1, 1, N.BC_ALL_BOUNDARY, cus=0, max_threads=256, cells=max(per, rows // 192))
            assert L, n
            check_tiles(L, 256)
            chunks = [window_rows(L, c) for c in range(L.g.nch)]
            assert 8 * max(chunks) <= 1 << 30, n
            assert sum(chunks) >= rows
    assert plan((1292,) * 3, 1, 1, N.BC_ALL_BOUNDARY, cus=0, max_threads=256, cells=16384) is None   # rows past 2^31
