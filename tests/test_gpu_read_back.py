"""Reading particle state back in pieces: every field equals what was set, for
counts around the piece boundaries (the staging holds 4 MiB: a read of all
fields of a few thousand particles is one piece, of 100k nine), and any
subset of fields."""
import numpy as np
import pytest

from mpm_amd import materials as mat
from mpm_amd.mesh import structured_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 1), (2, 1023), (3, 4096), (3, 58255), (2, 100003)])
@pytest.mark.parametrize("mc", [True, False])
def test_fields_come_back_as_set(dim, n, mc):
    from mpm_amd.capi import Solver
    r = np.random.default_rng(n + dim)
    coords, cells = structured_mesh((0.0,) * dim, (0.5,) * dim, (7, 5, 4)[:dim])
    s = Solver(dim, "usl")
    s.set_mesh(coords, cells)
    m = [mat.linear_elastic(1e6, 0.3, 1000.0)]
    if mc:
        m.append(mat.mohr_coulomb(1e6, 0.3, 1800.0, friction=30.0, dilation=0.0, cohesion=10.0))
    s.set_materials(np.stack(m))
    p = dict(x=r.uniform(0.01, 1.9, (n, dim)), u=r.normal(size=(n, dim)),
             v=r.normal(size=(n, dim)), stress=r.normal(size=(n, 6)),
             strain=r.normal(size=(n, 6)), F=r.normal(size=(n, 9)), mass=r.uniform(1, 2, n),
             volume=r.uniform(1, 2, n), density=r.uniform(1, 2, n),
             material_id=r.integers(0, len(m), n).astype(np.int32))
    sv = r.uniform(0.1, 1.0, (n, 9))
    s.set_particles(**p, statevars=sv)
    got = s.particles()
    for f in p:
        assert np.array_equal(got[f], p[f]), f
    is_mc = p["material_id"] == 1
    assert np.array_equal(got["statevars"][is_mc], sv[is_mc])
    assert not got["statevars"][~is_mc].any()
    cell = sum((p["x"][:, k] // 0.5).astype(int) * int(np.prod((7, 5, 4)[:k])) for k in range(dim))
    assert np.array_equal(got["cell"], cell) and got["cell"].dtype == np.int64
    c = coords[cells[cell]].mean(1)
    assert np.abs(got["xi"] - (p["x"] - c) / 0.25).max() < 1e-13
    some = s.particles(["F", "cell", "density"])
    for f in some:
        assert np.array_equal(some[f], got[f]), f


# One or two fields go straight to the arrays on a first read and where they take
# 1 to 4 MiB (or more, before the staging is made), others through pinned
# staging, which grows with them: 8192 particles in one piece of 3 MB, 30000 in
# three of 4 MiB, x and v of 120001 in 3D in two.
@pytest.mark.parametrize("dim,n", [(2, 1), (3, 257), (2, 8192), (3, 30000), (3, 120001)])
def test_reads_of_one_context_agree(dim, n):
    from mpm_amd.capi import Solver
    r = np.random.default_rng(n)
    coords, cells = structured_mesh((0.0,) * dim, (0.5,) * dim, (7, 5, 4)[:dim])
    p = dict(x=r.uniform(0.01, 1.9, (n, dim)), v=r.normal(size=(n, dim)),
             mass=r.uniform(1, 2, n), volume=r.uniform(1, 2, n), density=r.uniform(1, 2, n),
             material_id=r.integers(0, 2, n).astype(np.int32))
    reads = [["x", "v"], ["material_id", "cell", "density"], ["v"]]
    for first in range(3):
        s = Solver(dim, "usl")
        s.set_mesh(coords, cells)
        s.set_materials(np.stack([mat.linear_elastic(1e6, 0.3, 1000.0)] * 2))
        s.set_particles(**p)
        got = {}
        for k in range(3):
            f = reads[(first + k) % 3]
            some = s.particles(f)
            for a in f:
                if a in p:
                    assert np.array_equal(some[a], p[a]), (first, a)
                got.setdefault(a, some[a])
        all_ = s.particles()
        for a in got:
            assert np.array_equal(all_[a], got[a]) and all_[a].dtype == got[a].dtype, a
        s.close()
