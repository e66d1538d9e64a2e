"""Steps queued in blocks (graphs of several steps) against steps launched one
by one: same states bit for bit in ordered mode whatever the sizes of the
calls, the status of a call's last step, and a particle that leaves the mesh
inside a block, between blocks and in a call's last step.
"""
import numpy as np
import pytest

from mpm_amd import materials as mat
from mpm_amd import workloads

pytestmark = pytest.mark.gpu

FIELDS = ("x", "u", "v", "stress", "strain", "F", "volume", "density", "xi", "cell", "statevars")


def _deck(dim):
    if dim == 2:
        return workloads.collapse_2d(6, 9, 0.05, 1e6, 30.0, 1800.0, dt=1e-5)
    return workloads.collapse_3d(nx=8, ny=4, nz=4, block=(4, 4, 4))


@pytest.mark.parametrize("dim,ordered", [(2, True), (3, True), (2, False)])
def test_blocks_are_the_single_steps(dim, ordered):
    from mpm_amd.capi import Solver
    w = _deck(dim)
    a = w.setup(Solver(dim, w.scheme, ordered=ordered))
    b = w.setup(Solver(dim, w.scheme, ordered=ordered, graph=False))
    for calls in ((24,), (1, 3, 4, 5), (9, 20, 2), (8, 8, 31)):
        for n in calls:
            a.step(n, w.dt)
            b.step(n, w.dt)
            assert a.step_count == b.step_count
        pa, pb = a.particles(), b.particles()
        for f in FIELDS:
            if ordered:
                assert np.array_equal(pa[f], pb[f]), (f, calls)
            else:  # rounding of the atomic order over up to 115 steps
                s = max(float(np.abs(pb[f]).max()), 1e-300)
                assert np.abs(pa[f] - pb[f]).max() <= 1e-6 * s, (f, calls)


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("at", [1, 25, 26, 28, 29, 32, 40, 41])
def test_run_stops_at_the_step_a_particle_leaves(graph, at):
    """A free particle at constant velocity passes the mesh's side in step
    `at` of a 40 or 41 step run."""
    from mpm_amd.capi import Solver, UnlocatableParticle
    from mpm_amd.mesh import structured_mesh
    coords, cells = structured_mesh((0.0, 0.0), (1.0, 1.0), (4, 3))
    s = Solver(2, "usl", graph=graph)
    s.set_mesh(coords, cells)
    s.set_materials(mat.linear_elastic(1e3, 0.3, 1000.0)[None, :])
    s.set_gravity([0.0, 0.0])
    dt = 1e-3
    x = np.array([[4.0 - (at - 0.5) * dt, 1.5], [1.5, 1.5]])
    s.set_particles(x=x, mass=[250.0, 250.0], volume=[0.25, 0.25], density=[1000.0, 1000.0],
                    material_id=0, v=[[1.0, 0.0], [0.0, 0.0]])
    with pytest.raises(UnlocatableParticle) as e:
        for n in (24, 12, 4, 1):
            s.step(n, dt)
    assert "step %d" % (at - 1) in str(e.value)
    assert s.step_count == at
    p = s.particles(["x", "cell"])
    assert abs(p["x"][0, 0] - (4.0 + 0.5 * dt)) < 1e-9
    assert list(p["cell"] < 0) == [True, False]
