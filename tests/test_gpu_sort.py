"""The cell sort over its digit widths, passes, tile lengths and scan paths.

Ordered mode's gathers read each cell's particles from the sorted order (cell
ranges, ascending ids), fast mode only groups by it: particles in random order
over meshes of 2 to 1.2 million cells give the same step in both modes to
rounding only if the sort is a sort, and a second ordered run gives the same
bits.
"""
import numpy as np
import pytest

from mpm_amd import materials as mat
from mpm_amd.mesh import structured_mesh

pytestmark = pytest.mark.gpu


# cells 2 (1 digit), 1023 / 1024 (10 / 11 bits: 1 / 2 passes), 40k, 1.2M (21
# bits: 3 passes); particles around a wave, a tile, each tile length (64k, 512k,
# 2M), the table scanned in one workgroup and in tiles
@pytest.mark.parametrize("grid,n", [((2, 1), 300), ((33, 31), 1), ((33, 31), 255), ((32, 32), 257),
                                    ((200, 200), 65535), ((200, 200), 65536), ((33, 31), 70001),
                                    ((200, 200), 525001), ((1200, 1000), 40001),
                                    ((1200, 1000), 2100001)])
def test_ordered_step_from_random_order(grid, n):
    from mpm_amd.capi import Solver
    h = 0.1
    coords, cells = structured_mesh((0.0, 0.0), (h, h), grid)
    r = np.random.default_rng(n)
    x = r.uniform(1e-6, 1.0 - 1e-6, (n, 2)) * np.array(grid) * h
    v = r.uniform(-0.1, 0.1, (n, 2))
    out = []
    for ordered in (True, True, False):
        s = Solver(2, "usl", ordered=ordered)
        s.set_mesh(coords, cells)
        s.set_materials(mat.linear_elastic(1e6, 0.3, 1800.0)[None, :])
        s.set_gravity([0.0, -9.81])
        s.set_particles(x=x, v=v, mass=np.full(n, 1.8), volume=np.full(n, 1e-3),
                        density=np.full(n, 1800.0), material_id=0)
        s.step(2, 1e-5)
        out.append(s.particles(["x", "v", "stress", "cell"]))
        s.close()
    a, b, f = out
    for k in a:
        assert np.array_equal(a[k], b[k]), k
    assert np.array_equal(a["cell"], f["cell"])
    for k in ("x", "v", "stress"):  # sums of up to some 1000 terms in another order
        scale = max(float(np.abs(a[k]).max()), 1e-300)
        assert np.abs(a[k] - f[k]).max() <= 1e-11 * scale, k


# The sort by itself against numpy's stable one: digits of every width and 1 to
# 3 passes, and the three forms of the table scan: in one workgroup (up to 32768
# entries), in tiles that sum the totals before them, and with a scan of the
# totals (over 2048 tiles: 8.5 million keys with 10-bit digits).
@pytest.mark.parametrize("n,ncells", [
    (1, 1), (255, 2), (257, 1023), (4097, 1024), (8193, 40000), (65537, 1 << 20),
    (65537, 3), (300007, 1000), (525001, 1 << 20), (2097153, 5000000), (8500001, 700),
    (8500001, 700000)])
def test_sort_is_the_stable_sort(n, ncells):
    import ctypes as C
    from mpm_amd import capi
    lib = capi.load()  # its handle also finds the HIP runtime that it is linked to
    temp = lib["_ZN4mpmx20radix_sort_temp_intsEli"]
    temp.restype, temp.argtypes = C.c_int64, [C.c_int64, C.c_int]
    sort = lib["_ZN4mpmx18radix_sort_by_cellEPKiliPiS2_S2_P12ihipStream_t"]
    sort.restype = None
    sort.argtypes = [C.c_void_p, C.c_int64, C.c_int] + [C.c_void_p] * 4

    def hip(name, *args):
        assert lib[name](*args) == 0, name

    bufs = []

    def device(a):
        p = C.c_void_p()
        hip("hipMalloc", C.byref(p), C.c_size_t(a.nbytes))
        bufs.append(p)
        hip("hipMemcpy", p, C.c_void_p(a.ctypes.data), C.c_size_t(a.nbytes), 1)
        return p

    def host(p, a):
        hip("hipMemcpy", C.c_void_p(a.ctypes.data), p, C.c_size_t(a.nbytes), 2)
        return a

    # some particles in no cell: their key is ncells
    cell = np.random.default_rng(n).integers(-1, ncells + 2, n).astype(np.int32)
    key = np.where((cell >= 0) & (cell < ncells), cell, ncells).astype(np.int32)
    room = temp(n, ncells)
    # a margin on both sides of the temporaries tells of a write beyond them
    tmp = np.full(room + 2048, -7, np.int32)
    d_cell, d_tmp, d_keys, d_ids = device(cell), device(tmp), device(cell), device(cell)
    sort(d_cell, n, ncells, d_keys, d_ids, d_tmp.value + 4 * 1024, None)
    hip("hipDeviceSynchronize")
    keys, ids, tmp = host(d_keys, np.empty_like(cell)), host(d_ids, np.empty_like(cell)), host(d_tmp, tmp)
    for p in bufs:
        hip("hipFree", p)
    order = np.argsort(key, kind="stable")
    assert np.array_equal(ids, order)
    assert np.array_equal(keys, key[order])
    assert np.all(tmp[:1024] == -7) and np.all(tmp[1024 + room:] == -7)
