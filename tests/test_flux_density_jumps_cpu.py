"""CPU check of the stage kernels' Roe flux (famrdp_math.h roe_flux2, compiled
for the host) on faces between states of very different density, either side
the lighter one, against flux/roe.py:21-85 in extended precision.

Tolerance: the flux is about 140 operations none of which cancels terms much
larger than the largest flux component, so its error is a few tens of roundings
of that component: 64 of 2^-53."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle import numerics as ON

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "famrdp-jax_amd", "csrc")
G = 1.4
TOL = 64 * 2.0 ** -53


@pytest.fixture(scope="module")
def hc(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("fhc") / "libfhc.so")
    subprocess.run([hipcc, "--cuda-host-only", "-O1", "-ffp-contract=off", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                    os.path.join(HERE, "hostcheck", "flux_hostcheck.hip"), "-o", out],
                   check=True, capture_output=True)
    return ctypes.CDLL(out)


def faces(ratio, n, seed):
    """States of pressure about 1 and |u| < 0.5, left density `ratio` times the right one, and area vectors."""
    rng = np.random.default_rng(seed)
    side = lambda s: np.stack([s * rng.uniform(0.8, 1.2, n), *(rng.uniform(-0.5, 0.5, n) for _ in range(3)),  # noqa: E731
                               rng.uniform(0.9, 1.1, n)], axis=1)
    return side(min(ratio, 1.0)), side(min(1.0 / ratio, 1.0)), rng.uniform(-1, 1, (n, 3))


RATIOS = [1e-6, 1e-4, 1e-3, 1e-2, 1.0, 1e2, 1e3, 1e4, 1e6]


@pytest.mark.parametrize("full", [0, 1])
@pytest.mark.parametrize("ratio", RATIOS)
def test_flux_between_light_and_heavy(hc, ratio, full):
    n = 500
    pl, pr, S = faces(ratio, n, 31)
    F = np.zeros((n, 5))
    P = lambda a: np.ascontiguousarray(a).ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    hc.hc_roe_flux2(n, full, P(pl), P(pr), P(S), ctypes.c_double(G), P(F))
    x = lambda a: a.T.astype(np.longdouble)  # noqa: E731
    g = np.longdouble(G)
    A = np.sqrt((x(S) ** 2).sum(axis=0))
    ref = (2 * A * ON.roe_flux(ON.prim_to_cons(x(pl), g), ON.prim_to_cons(x(pr), g), x(S) / A, gamma=g)).T
    err = np.abs(F - ref).max(axis=1) / np.abs(ref).max(axis=1)
    print(f"ratio {ratio:g}: max {float(err.max()):.2e}")
    assert float(err.max()) <= TOL
