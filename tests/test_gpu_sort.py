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
# 2M) and both scan paths
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
