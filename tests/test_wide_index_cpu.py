"""CPU check of the wide stage kernel's slot maps (WideGeom in famrdp_tiles.h):
the branch-free cell, tensor and face maps against FusedGeom's, every step map
against the neighbour it is read for."""
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
    out = str(tmp_path_factory.mktemp("wide") / "libwide.so")
    subprocess.run([hipcc, "--cuda-host-only", "-O2", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                    os.path.join(HERE, "hostcheck", "wide_index_hostcheck.hip"), "-o", out],
                   check=True, capture_output=True)
    lib = ctypes.CDLL(out)
    lib.wide_bad.restype = ctypes.c_int64
    return lib


@pytest.mark.parametrize("shape", [(3, 4, 4), (4, 4, 8), (4, 8, 8), (3, 4, 5)])
def test_wide_slot_maps(hc, shape):
    assert hc.wide_bad(*shape) == 0
