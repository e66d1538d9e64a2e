"""Fast mode's inverse of the hex8 map against ordered mode's (the reference's
iteration step by step) over cell sizes and distortions.

The iteration contracts by 1 - h/2 per step, so the size decides which part
of the fast form answers: small cells (thousands of steps, taken by powers of
the step), cells of metres (a few steps), cells whose full step overshoots
(line search: the general loop).
"""
import numpy as np
import pytest

from mpm_amd import materials as mat
from mpm_amd import workloads

pytestmark = pytest.mark.gpu


def _deck(h, drape, warp):
    w = workloads.collapse_3d(nx=7, ny=5, nz=6, h=h, block=(6, 5, 5), dt=1e-6 * h / 0.01)
    w.materials = mat.linear_elastic(1e6, 0.3, 1800.0)[None, :]
    X = w.coords
    u = X / X.max(0)
    X[:, 2] *= 1.0 + drape * u[:, 0] - 0.5 * drape * u[:, 1]
    bump = np.prod(np.sin(np.pi * u), axis=1)
    for k in range(3):
        X[:, k] += warp * h * bump * np.cos((k + 1) * np.pi * u[:, (k + 1) % 3])
    w.isoparametric = True
    return w


@pytest.mark.parametrize("h", [0.002, 0.01, 0.1, 0.5, 2.0, 6.0])
@pytest.mark.parametrize("drape,warp", [(0.0, 0.0), (0.02, 0.0), (0.3, 0.0), (0.3, 0.25)])
def test_fast_inverse_ends_where_the_iteration_does(h, drape, warp):
    from mpm_amd.capi import Solver
    w = _deck(h, drape, warp)
    p = {}
    for ordered in (True, False):
        s = w.setup(Solver(3, "musl", ordered=ordered))
        r = np.random.default_rng(3)
        # some particles cross a face within the steps
        s.assign_velocity(r.uniform(-1.0, 1.0, (s.nparticles, 3)) * 0.05 * h / w.dt)
        s.step(4, w.dt)
        p[ordered] = s.particles(["x", "xi", "cell"])
    assert np.array_equal(p[True]["cell"], p[False]["cell"])
    d = np.abs(p[True]["xi"] - p[False]["xi"]).max(1)
    # a residual within rounding of 1e-10 may take one step (1e-10 at most)
    # more or less; the others differ by rounding and the 2e-13 the fast form
    # neglects. Velocities move particles by up to 0.1 h against each other in
    # a step, so 4 steps at local coordinates 1.5e-10 apart displace by 6e-11 h.
    dx = np.abs(p[True]["x"] - p[False]["x"]).max()
    assert dx <= 6e-11 * h
    close = d <= 1e-12 + 4.0 * 2.3e-16 * np.abs(w.coords).max() / h
    assert np.mean(close) > 0.99, (np.mean(close), d.max())
    assert d.max() <= 1.5e-10, d.max()
