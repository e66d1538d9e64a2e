"""Ordered mode's node sums at the edges of their windows.

A node's particles are summed in ascending id order, 64 ranks at a time, by a
wave up to 128 particles and by one lane beyond; MUSL's momentum sums take the
ranks from the force sums. The oracle adds the same terms in the same order:
the results have to be the same bits.
"""
import numpy as np
import pytest

import oracle
from mpm_amd import materials as mat
from mpm_amd.mesh import structured_mesh

pytestmark = pytest.mark.gpu


# 2 cells a side: the central node holds all n particles, the others fewer
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("scheme", ["musl", "usl", "usf"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 200])
def test_node_sums_are_the_oracles_bits(dim, scheme, n):
    from mpm_amd.capi import Solver
    h = 0.1
    coords, cells = structured_mesh((0.0,) * dim, (h,) * dim, (2,) * dim)
    r = np.random.default_rng(n)
    x = r.uniform(0.2 * h, 1.8 * h, (n, dim))
    v = r.uniform(-0.1, 0.1, (n, dim))
    out = []
    for s in (Solver(dim, scheme, ordered=True), oracle.Oracle(dim, scheme)):
        s.set_mesh(coords, cells)
        s.set_materials(mat.linear_elastic(1e6, 0.3, 1800.0)[None, :])
        s.set_gravity([0.0] * (dim - 1) + [-9.81])
        s.set_particles(x=x, v=v, mass=np.full(n, 1.8), volume=np.full(n, 1e-3),
                        density=np.full(n, 1800.0), material_id=0)
        s.step(4, 1e-5)
        out.append(s.particles(["x", "v", "stress", "cell"]))
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k
