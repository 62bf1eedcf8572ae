"""CPU check of the inviscid RHS kernel's slot maps (CrossGeom in famrdp_tiles.h):
every staged cell has one slot, every cell a face reads is found in its own."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "famrdp-jax_amd", "csrc")


@pytest.fixture(scope="module")
def hc(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("cross") / "libcross.so")
    subprocess.run([hipcc, "--cuda-host-only", "-O2", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                    os.path.join(HERE, "hostcheck", "cross_index_hostcheck.hip"), "-o", out],
                   check=True, capture_output=True)
    lib = ctypes.CDLL(out)
    lib.cross_bad.restype = ctypes.c_int64
    return lib


@pytest.mark.parametrize("shape", [(4, 4, 4), (3, 4, 5)])
def test_cross_slot_maps(hc, shape):
    assert hc.cross_bad(*shape) == 0
