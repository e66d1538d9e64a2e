"""Fast mode's stress update (regrouped arithmetic, return mappings compacted
per workgroup) against ordered mode's, which the parity tests tie to the
oracle bit for bit: one step from the same random state.

Counts at the edges of a wave and of a workgroup (128 and 256 particles);
materials side by side: linear elastic, cohesionless, cohesive with dilation
and tension cutoff, softening; box cells (gradients axis by axis) and sheared
ones (general Jacobian); stresses inside, on and outside the surface, some with
two equal principal values (a corner of the surface, where the Lode angle's
derivative is singular).
"""
import numpy as np
import pytest

from mpm_amd import materials as mat
from mpm_amd.mesh import structured_mesh

pytestmark = pytest.mark.gpu

FIELDS = ("x", "v", "stress", "strain", "F", "volume", "density", "xi", "statevars")


def _materials():
    return np.stack([
        mat.mohr_coulomb(5e6, 0.3, 1800.0, friction=30.0, dilation=0.0, cohesion=0.0),
        mat.linear_elastic(4e6, 0.25, 1700.0),
        mat.mohr_coulomb(3e6, 0.2, 2000.0, friction=35.0, dilation=5.0, cohesion=800.0,
                         tension_cutoff=300.0),
        mat.mohr_coulomb(4e6, 0.3, 1900.0, friction=32.0, dilation=3.0, cohesion=500.0,
                         residual_friction=25.0, residual_dilation=0.0, residual_cohesion=100.0,
                         peak_pdstrain=0.0, residual_pdstrain=1e-2, softening=True)])


def _state(dim, n, shear, seed):
    r = np.random.default_rng(seed)
    h, nc = 0.1, (5, 4) if dim == 2 else (4, 3, 3)
    coords, cells = structured_mesh((0.0,) * dim, (h,) * dim, nc)
    pick = r.integers(0, len(cells), n)
    x = coords[cells[pick][:, 0]] + h * r.uniform(0.05, 0.95, (n, dim))
    if shear:
        coords = coords.copy()
        coords[:, 0] += 0.2 * coords[:, dim - 1]
        x[:, 0] += 0.2 * x[:, dim - 1]
    mid = r.integers(0, 4, n)
    s = np.zeros((n, 6))
    p = -np.exp(r.uniform(np.log(50.0), np.log(2e4), n))
    k = r.uniform(0.2, 1.0, (n, 2))
    s[:, dim - 1] = p
    s[:, (dim) % 3], s[:, (dim + 1) % 3] = p * k[:, 0], p * k[:, 1]
    s[::5, (dim + 1) % 3] = s[::5, dim % 3]  # two equal principal stresses
    s[:, 3] = r.uniform(-0.2, 0.2, n) * p
    s[::5, 3] = 0.0
    if dim == 3:
        s[:, 4:] = r.uniform(-0.1, 0.1, (n, 2)) * p[:, None]
        s[::5, 4:] = 0.0
    s[3::7, :3] = r.uniform(5.0, 400.0, (len(s[3::7]), 3))  # tension
    s[3::7, 3:] *= 0.01
    if dim == 2:
        s[3::7, 4:] = 0.0
    rho = _materials()[mid, 1]
    vol = np.full(n, (h ** dim) / 8)
    v = r.uniform(-0.05, 0.05, (n, dim))
    return coords, cells, dict(x=x, v=v, stress=s, mass=vol * rho, volume=vol, density=rho,
                               material_id=mid)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("scheme", ["usf", "usl", "musl"])
@pytest.mark.parametrize("shear", [False, True])
@pytest.mark.parametrize("n", [1, 63, 128, 129, 257, 1000])
def test_fast_step_is_the_ordered_step(dim, scheme, shear, n):
    from mpm_amd.capi import Solver
    coords, cells, state = _state(dim, n, shear, seed=n + dim)
    out = {}
    for ordered in (True, False):
        s = Solver(dim, scheme, ordered=ordered)
        # the sheared mesh is located by the inverse element map
        s.set_mesh(coords, cells, isoparametric=shear)
        s.set_materials(_materials())
        s.set_gravity([0.0] * (dim - 1) + [-9.81])
        s.set_particles(**state)
        s.step(1, 2e-5)
        out[ordered] = s.particles()
        s.close()
    a, b = out[True], out[False]
    assert np.array_equal(a["cell"], b["cell"])
    if n >= 128:
        y = a["statevars"][:, 0]
        assert np.any(y == 0) and np.any(y == 1) and np.any(y == 2)
    assert np.array_equal(a["statevars"][:, 0], b["statevars"][:, 0])
    # fast mode's bar per step, 1e-12 of the field's largest value. A return of
    # several corrections from far outside the surface magnifies rounding, by
    # up to 1e5 in these states (the reference's arithmetic, its inputs moved by
    # an ulp, moves its results as far): 1e5 * 2.2e-16 and a factor of 4
    for f in FIELDS:
        scale = max(float(np.abs(a[f]).max()), 1e-300)
        d = np.abs(a[f] - b[f]).reshape(n, -1).max(1) / scale
        assert d.max() <= 1e-10, (f, d.max())
        assert np.mean(d <= 1e-12) >= 0.995, (f, np.sort(d)[-4:])


def _one_step(coords, cells, state, materials, scheme, iso=False, vu="flip", g=9.81):
    from mpm_amd.capi import Solver
    out = {}
    for ordered in (True, False):
        s = Solver(3, scheme, vu, ordered=ordered)
        s.set_mesh(coords, cells, isoparametric=iso)
        s.set_materials(materials)
        s.set_gravity([0.0, 0.3 * g, -g])
        s.set_particles(**state)
        s.step(1, 2e-5)
        out[ordered] = s.particles()
        s.close()
    return out[True], out[False]


def _compare(a, b, extra=0.0):
    n = len(a["x"])
    assert np.array_equal(a["cell"], b["cell"])
    assert np.array_equal(a["statevars"][:, 0], b["statevars"][:, 0])
    for f in FIELDS:
        scale = max(float(np.abs(a[f]).max()), 1e-300)
        d = np.abs(a[f] - b[f]).reshape(n, -1).max(1) / scale
        assert d.max() <= 1e-10 + extra, (f, d.max())
        assert np.mean(d <= 1e-12 + extra) >= 0.995, (f, np.sort(d)[-4:])


# Box cells of three different sides: a side or a component taken for another
# shows. One node moved by 3 % of a side: no cell is treated as a box then (the
# flag is the mesh's), and the general kernels run on a Cartesian mesh.
@pytest.mark.parametrize("scheme", ["usf", "usl", "musl"])
@pytest.mark.parametrize("vu", ["flip", "apic"])
@pytest.mark.parametrize("move", [False, True])
def test_unequal_sides(scheme, vu, move):
    h = np.array([0.1, 0.07, 0.13])
    coords, cells, state = _state(3, 1000, False, seed=5)
    coords, state["x"] = coords / 0.1 * h, state["x"] / 0.1 * h
    state["volume"] = state["volume"] / 0.1**3 * h.prod()
    state["mass"] = state["volume"] * state["density"]
    if move:
        centre = int(np.argmin(np.abs(coords - coords.mean(0)).sum(1)))
        coords[centre] += 0.03 * h * np.array([1.0, -1.0, 1.0])
    a, b = _one_step(coords, cells, state, _materials(), scheme, vu=vu)
    _compare(a, b)


# Coordinates far from the origin. Sides of 1/16 m, an offset of 2^17 m and
# positions on a grid of 2^-30 m are exact in 64 bits, so the step there is the
# step at the origin but for rounding of the coordinates' products: the Jacobian
# of 8 products of offset size, 8 * 2^-53 * 2^17 / (1 / 32) of its entries in
# ordered mode, which the return mappings magnify by up to 10. The boxes' sides
# do not see the offset: fast mode is no further from the step at the origin
# than ordered mode.
@pytest.mark.parametrize("scheme", ["usf", "usl", "musl"])
def test_large_coordinates(scheme):
    h, off = 0.0625, 2.0**17
    coords, cells, state = _state(3, 600, False, seed=6)
    coords = np.round(coords / 0.1) * h
    state["x"] = np.round(state["x"] / 0.1 * h * 2.0**30) / 2.0**30
    at0, _ = _one_step(coords, cells, state, _materials(), scheme)
    state["x"] = state["x"] + off
    a, b = _one_step(coords + off, cells, state, _materials(), scheme)
    assert np.array_equal(a["cell"], b["cell"])
    bound = 10 * 8 * 2.0**-53 * off * 32
    for f in ("v", "stress", "strain", "F", "volume"):
        scale = max(float(np.abs(at0[f]).max()), 1e-300)
        ea, eb = (float(np.abs(q[f] - at0[f]).max()) / scale for q in (a, b))
        assert ea <= bound and eb <= bound, (f, ea, eb, bound)
        assert eb <= ea + 1e-10, (f, ea, eb)


# Softening and separation. Plastic strains below, between and above the peak
# and residual ones, in materials with and without tension cutoff, and particles
# below the critical density.
@pytest.mark.parametrize("scheme", ["usf", "usl", "musl"])
@pytest.mark.parametrize("n", [129, 1000])
def test_softened_and_separated_particles(scheme, n):
    soft = dict(residual_friction=25.0, residual_dilation=1.0, residual_cohesion=100.0,
                peak_pdstrain=1e-3, residual_pdstrain=1e-2, softening=True,
                packing_fraction=0.6, packing_fraction_minimum=0.5)
    materials = np.stack([
        mat.mohr_coulomb(4e6, 0.3, 1900.0, friction=32.0, dilation=3.0, cohesion=500.0, **soft),
        mat.linear_elastic(4e6, 0.25, 1700.0),
        mat.mohr_coulomb(3e6, 0.2, 2000.0, friction=35.0, dilation=5.0, cohesion=800.0,
                         tension_cutoff=1200.0, **soft),
        mat.mohr_coulomb(3e6, 0.2, 2000.0, friction=35.0, dilation=5.0, cohesion=800.0,
                         tension_cutoff=300.0, packing_fraction=0.6,
                         packing_fraction_minimum=0.5)])
    coords, cells, state = _state(3, n, False, seed=7)
    r = np.random.default_rng(8)
    mid = state["material_id"]
    rho = materials[mid, 1] * np.where(np.arange(n) % 11 == 3, 0.8, 1.0)
    pds = r.choice([0.0, 5e-4, 2e-3, 9e-3, 1e-2, 3e-2], n)
    sv = np.zeros((n, mat.NSTATEVARS))
    sv[:, 1:5] = np.stack([np.radians(materials[mid, 4]), np.radians(materials[mid, 5]),
                           materials[mid, 6], materials[mid, 12]], 1)
    sv[:, 8] = pds
    state.update(density=rho, mass=state["volume"] * rho, statevars=sv)
    a, b = _one_step(coords, cells, state, materials, scheme)
    y, mc = a["statevars"][:, 0], materials[mid, 0] == 1
    between = (pds > 1e-3) & (pds < 1e-2) & mc & (mid != 3)
    assert np.any(y == 3)
    assert np.any(between & (y == 1)) and np.any(between & (y == 2))  # a softening modulus
    assert np.any((pds >= 1e-2) & (mid == 0) & (y == 1))              # residual strength
    assert np.any(np.abs(a["statevars"][between, 1] - sv[between, 1]) > 1e-3)
    cut = between & (mid == 2)
    assert np.any(a["statevars"][cut, 4] < 1200.0)  # the apex of the softened cone
    _compare(a, b)
