"""What a read of the particle state allocates (recorded calls of the host
code, no GPU): a context's first read of a few components makes no staging,
which a program that reads once would pay for; later reads keep one."""
import pytest

import hip_record


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return hip_record.build(tmp_path_factory.mktemp("hip"))


@pytest.mark.parametrize("dim,n", [(2, 8192), (3, 60000)])
def test_first_read_of_few_components_makes_no_staging(lib, dim, n):
    out = hip_record.run(lib, """
dim, n = %d, %d
p0 = rec.hip_record_pinned_bytes()
s = solver(dim, "usl", n)
p1 = rec.hip_record_pinned_bytes()
s.particles(["x", "v"])
first = log()
assert first == ["to_host %%d" %% (n * 8)] * (2 * dim), first
s.particles(["x", "v"])
assert any(l.startswith("pinned") for l in log())
for _ in range(3):
    s.particles(["x", "v"])
    later = log()
    assert not [l for l in later if l.startswith(("malloc", "pinned"))], later
s.particles()
assert rec.hip_record_pinned_bytes() - p1 <= 8 << 20
s.close()
assert rec.hip_record_pinned_bytes() == p0
print("ok")
""" % (dim, n))
    assert "ok" in out


# small reads, reads of many components and large ones gain from the first on
@pytest.mark.parametrize("dim,n,fields", [(2, 512, ["x", "v"]), (3, 8192, None),
                                          (3, 1000000, ["x", "v"])])
def test_first_read_packs_where_that_is_faster(lib, dim, n, fields):
    out = hip_record.run(lib, """
s = solver(%d, "usl", %d)
fields = %r
s.particles(fields) if fields else s.particles()
assert any("k_pack_rows" in l for l in log())
print("ok")
""" % (dim, n, fields))
    assert "ok" in out
