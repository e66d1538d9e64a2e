"""Fast mode's inverse of the hex8 map (mpm_amd/csrc/mpmx_device.h), compiled
for the host, against the general loop over cell sizes, distortions and points
inside, near and far from the cell.

The loop stops within 1e-10 of the solution's residual, so the two may end one
step of at most 1e-10 apart: 2e-10 with the rounding of that test. In strongly
distorted cells single steps of the loop would increase the residual and are
halved: fast mode must not take such steps at once."""
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
    exe = str(tmp_path_factory.mktemp("iso") / "iso_hex_check")
    subprocess.run([CLANG, "-O2", "-std=c++17", "-ffp-contract=off", "-mfma",
                    "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I", CSRC,
                    os.path.join(HERE, "host", "iso_hex_check.cpp"), "-o", exe], check=True)

    def run(seed, points, h, distortion):
        out = subprocess.run([exe, str(seed), str(points), str(h), str(distortion)], check=True,
                             capture_output=True, text=True).stdout.split()
        return [int(v) for v in out[:3]] + [float(out[3]), int(out[4])]
    return run


# the last three: seeds of the strongest distortion where some steps increase
# the residual
@pytest.mark.parametrize("h,distortion,seed,points", [
    (0.001, 0.02, 1, 300), (0.002, 0.4, 1, 300), (0.01, 0.02, 1, 2000), (0.01, 0.4, 1, 2000),
    (0.1, 0.25, 1, 5000), (0.5, 0.6, 1, 5000), (1.9, 0.4, 1, 5000), (4.0, 0.1, 1, 5000),
    (0.7, 0.9, 5, 60000), (0.7, 0.9, 6, 60000), (1.5, 0.9, 8, 60000)])
def test_fast_inverse_is_the_general_loops(check, h, distortion, seed, points):
    n, general, differing, worst, _ = check(seed, points, h, distortion)
    assert n > points // 2
    assert differing == 0
    assert worst <= 2e-10, worst


# A search for the number of steps to jump is up to 14 squarings of the step's
# matrix. Cells of some mm reach the loop's limit of 10000 steps first: 12
# searches of up to 15 octaves a point, not one every 16 steps.
@pytest.mark.parametrize("h", [0.0005, 0.001, 0.002, 0.003, 0.005])
@pytest.mark.parametrize("distortion", [0.02, 0.1, 0.4, 0.6])
def test_refused_jumps_are_not_sought_again_and_again(check, h, distortion):
    n, general, differing, worst, octaves = check(1, 300, h, distortion)
    assert differing == 0 and worst <= 2e-10
    assert octaves <= 12 * 15, octaves
