"""Device memory of a context and of the step without allocation (recorded
calls of the host code, no GPU)."""
import pytest

import hip_record


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return hip_record.build(tmp_path_factory.mktemp("hip"))


def test_deferred_list_only_where_returns_are_deferred(lib):
    """3D fast mode returns its yielding particles in the stress kernels: a
    Mohr-Coulomb context holds 9 state variables a particle more than a linear
    elastic one; 2D and ordered mode also the list (4 bytes) and its records
    (14 doubles)."""
    out = hip_record.run(lib, """
def held(dim, ordered, mc, n=4096):
    p0 = rec.hip_record_device_bytes()
    s = solver(dim, "musl", n, mc=mc, ordered=ordered)
    out = rec.hip_record_device_bytes() - p0
    s.close()
    return out
n = 4096
for dim, ordered, more in ((3, False, 72), (3, True, 188), (2, False, 188), (2, True, 188)):
    assert held(dim, ordered, True) - held(dim, ordered, False) == more * n, (dim, ordered)
print("ok")
""")
    assert "ok" in out


def test_noalloc_step_takes_3d_decks_of_its_size(lib):
    """64 MiB of scratch at 22 bytes a particle (keys, order, scan list and the
    sort's 10 bytes) hold 2 million 3D Mohr-Coulomb particles in fast mode."""
    out = hip_record.run(lib, """
s = solver(3, "musl", 2000000)
s.step_noalloc(1, 1e-6)
assert any("k_stress_fast" in l for l in log())
print("ok")
""")
    assert "ok" in out


def test_backward_pass_holds_no_more_for_its_plastic_list(lib):
    """The backward pass's list: ids, apex flags and 6 columns a particle; its
    12 output columns lie in the forward step's records of deferred returns,
    or, in 3D fast mode, which has no such records, in columns of their own
    (fewer than those records' 14)."""
    out = hip_record.run(lib, """
n = 4096
for dim, ordered, mc, cols in ((2, False, True, 6), (2, True, True, 6), (3, True, True, 6),
                               (3, False, True, 18), (3, False, False, 6)):
    s = solver(dim, "musl", n, mc=mc, ordered=ordered)
    s.adjoint_forward(4, 1e-6, checkpoint_every=2)
    log()
    p0 = rec.hip_record_device_bytes()
    s.adjoint_backward(dL_dx=np.ones((n, dim)))
    nodes = (2 + 8 * dim) * s.nnodes * 8
    parts = (3 * dim + 10) * n * 8
    held = rec.hip_record_device_bytes() - p0 - nodes - parts - (2 + 2 * n) * 4
    assert held == cols * n * 8, (dim, ordered, held / n / 8)
    s.close()
print("ok")
""")
    assert "ok" in out
