"""CPU check of the reverse sweeps' tables (famrdp_reverse.h): for blocks of
any size and any number of waves a GPU holds, every cell of every block
belongs to exactly one tile, and a tile's planes and lanes lie in its block.
The header is compiled for the host into a test-only library."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "famrdp-jax_amd", "csrc")
ip = ctypes.POINTER(ctypes.c_int32)


@pytest.fixture(scope="module")
def hc(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("stc") / "libstc.so")
    subprocess.run([hipcc, "--cuda-host-only", "-O2", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                    os.path.join(HERE, "hostcheck", "sweep_tiles_hostcheck.hip"), "-o", out],
                   check=True, capture_output=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("lanes", [58, 60, 64])
@pytest.mark.parametrize("slots", [8, 2048])
def test_tables_cover_every_cell_once(hc, lanes, slots):
    planes = np.array([4, 5, 36, 100, 7, 33], dtype=np.int32)
    cells = np.array([16, 58, 59, 129, 1, 640], dtype=np.int32)
    cap = 1 << 16
    out = np.zeros(4 * cap, dtype=np.int32)
    n = hc.sweep_table(len(planes), planes.ctypes.data_as(ip), cells.ctypes.data_as(ip), lanes,
                       ctypes.c_int64(slots), cap, out.ctypes.data_as(ip))
    assert n > 0
    seen = [np.zeros((p, c), dtype=int) for p, c in zip(planes, cells)]
    for b, p0, p1, base in out[:4 * n].reshape(n, 4):
        assert 0 <= p0 < p1 <= planes[b] and 0 <= base < cells[b]
        seen[b][p0:p1, base:base + lanes] += 1
    assert all((s == 1).all() for s in seen)
