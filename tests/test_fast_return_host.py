"""3D fast mode's constitutive update (mpm_amd/csrc/mpmx_fast.h), compiled for
the host, against the reference's arithmetic (mpmx_device.h) on random states.

The two group the same sums differently, so a returned stress differs by what
rounding leaves, magnified by the return: no more than moving the start stress
by one ulp moves the reference's own result, and a few ulp of the stresses (up
to 2e4 Pa: 3.6e-12 Pa) in the mean. Yield states, softened strengths and plastic
strains are the same."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "mpm_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CLANG = os.path.join(ROCM, "llvm", "bin", "clang++")

pytestmark = pytest.mark.skipif(not os.path.exists(CLANG), reason="needs ROCm's clang++")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ret") / "fast_return_check")
    subprocess.run([CLANG, "-O2", "-std=c++17", "-ffp-contract=off", "-mfma",
                    "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I", CSRC,
                    os.path.join(HERE, "host", "fast_return_check.cpp"), "-o", exe], check=True)

    def run(*args):
        out = subprocess.run([exe] + [str(a) for a in args], check=True, capture_output=True,
                             text=True).stdout.split()
        return [int(v) for v in out[:7]] + [float(v) for v in out[7:]]
    return run


@pytest.mark.parametrize("softening", [0, 1])
def test_update_is_the_references(check, softening):
    n, elastic, shear, tensile, separated, softened, mismatches, mean, most, nudge = \
        check(1, 200000, softening)
    assert min(elastic, shear, tensile, separated) > 5000
    assert (softened > 5000) == bool(softening)
    assert mismatches == 0
    assert mean <= 4 * 3.6e-12 and most <= nudge, (mean, most, nudge)
