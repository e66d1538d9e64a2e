"""Runs a piece of Python against libmpmx.so with the recording stand-in for
the HIP runtime (host/hip_record.cpp) in a process of its own: what the host
code allocates, copies and launches, without a GPU."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
rec = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
rec.hip_record_log.restype = ctypes.c_char_p
rec.hip_record_device_bytes.restype = ctypes.c_size_t
rec.hip_record_pinned_bytes.restype = ctypes.c_size_t
def log():
    out = rec.hip_record_log().decode().split("\\n")[:-1]
    rec.hip_record_clear()
    return out
import numpy as np
from mpm_amd import materials as mat
from mpm_amd import capi
from mpm_amd.mesh import structured_mesh
from mpm_amd.capi import Solver
# no kernel runs, so no particle is located: entry points that use the cells on
# the host (generate_gauss, compute_volume_mass) are not for here
def solver(dim, scheme, n, mc=True, grid=None, **kw):
    coords, cells = structured_mesh((0.,) * dim, (0.5,) * dim, grid or (8, 4, 4)[:dim])
    s = Solver(dim, scheme, **kw)
    s.set_mesh(coords, cells)
    m = mat.linear_elastic(1e6, 0.3, 1800.0)
    if mc:
        m = mat.mohr_coulomb(1e6, 0.3, 1800.0, friction=30.0, dilation=0.0, cohesion=10.0)
    s.set_materials(m[None, :])
    s.set_particles(x=np.full((n, dim), 0.3), mass=np.ones(n), volume=np.ones(n),
                    density=np.ones(n), material_id=0)
    log()
    return s
"""


def build(directory):
    lib = os.path.join(str(directory), "libhip_record.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(HERE, "host", "hip_record.cpp"), "-o", lib], check=True)
    return lib


def run(lib, code):
    env = dict(os.environ, PYTHONPATH=os.path.dirname(HERE))
    p = subprocess.run([sys.executable, "-c", PRELUDE + code, lib], env=env, text=True,
                       capture_output=True, timeout=110)
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout
