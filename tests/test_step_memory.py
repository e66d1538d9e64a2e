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
