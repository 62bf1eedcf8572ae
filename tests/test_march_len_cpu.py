"""The marching kernel's segment length: near the variant's, and of those the
one whose rounds of workgroups times planes are fewest (recomputed here)."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "famrdp-jax_amd", "csrc")


@pytest.fixture(scope="module")
def hc(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("mlen") / "libmlen.so")
    subprocess.run([hipcc, "--cuda-host-only", "-O2", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                    os.path.join(HERE, "hostcheck", "march_len_hostcheck.hip"), "-o", out],
                   check=True, capture_output=True)
    return ctypes.CDLL(out)


def _tiles(nj, nk, tj, tk):
    full, r = divmod(nk, tk)
    strips = -(-nj // tk) * -(-r // tj)
    ntj = -(-nj // tj)
    return ntj * full + strips if tj != tk and r and strips < ntj else ntj * -(-nk // tk)


def _cost(dims, length, tj, tk, slots):
    segs = [-(-d[0] // length) for d in dims]
    wgs = sum(n * _tiles(d[1], d[2], tj, tk) for n, d in zip(segs, dims))
    return -(-wgs // slots) * (max(-(-d[0] // n) for n, d in zip(segs, dims)) + 3.5), wgs


@pytest.mark.parametrize("dims", [[(4, 4, 4)], [(124, 124, 124)], [(100, 100, 100)], [(7, 40, 300)], [(300, 9, 70)],
                                  [(60, 52, 84), (20, 90, 33), (96, 17, 64)]])
@pytest.mark.parametrize("tj,tk,L", [(16, 16, 32), (8, 32, 20), (8, 32, 32), (8, 32, 52), (8, 32, 10)])
def test_length_of_fewest_rounds(hc, dims, tj, tk, L):
    flat = np.array(dims, dtype=np.int32).reshape(-1)
    units, wgs = ctypes.c_double(), ctypes.c_int64()
    got = hc.len_of(tj, tk, L, len(dims), flat.ctypes.data_as(ctypes.c_void_p), 512, ctypes.byref(units),
                    ctypes.byref(wgs))
    allowed = range(-(-7 * L // 10), 14 * L // 10 + 1)
    assert got in allowed
    assert (units.value, wgs.value) == _cost(dims, got, tj, tk, 512)
    assert units.value == min(_cost(dims, x, tj, tk, 512)[0] for x in allowed)
