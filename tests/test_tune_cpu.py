"""CPU check of the autotuner's choice (famrdp_tune.h): one disturbed launch pair,
whichever it is, does not drop the best variant; variants that do not fit are
never timed; ties keep the earlier variant."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "famrdp-jax_amd", "csrc")


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("thc") / "libthc.so")
    subprocess.run([hipcc, "--cuda-host-only", "-O1", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                    os.path.join(HERE, "hostcheck", "tune_hostcheck.hip"), "-o", out], check=True, capture_output=True)
    lib = ctypes.CDLL(out)

    def choose(cold, warm, more, fits=None, reps=3):
        n = len(cold)
        f = lambda a, t: np.ascontiguousarray(a, dtype=t)  # noqa: E731
        arr = [f(fits if fits is not None else [True] * n, np.bool_)] + [f(a, np.float32) for a in (cold, warm, more)]
        ms = np.zeros(n, dtype=np.float32)
        P = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
        return lib.hc_tune(n, P(arr[0]), reps, P(arr[1]), P(arr[2]), P(arr[3]), P(ms)), ms
    return choose


TIMES = np.array([2.2, 1.3, 1.0, 1.6, 1.2])


@pytest.mark.parametrize("pair", ["cold", "warm"])
@pytest.mark.parametrize("by", [1.6, 30.0])
def test_one_disturbed_pair_does_not_drop_the_best(choose, pair, by):
    cold, warm = 1.05 * TIMES, TIMES.copy()
    (cold if pair == "cold" else warm)[2] *= by
    best, ms = choose(cold, warm, TIMES)
    assert best == 2 and ms[2] < 1.1


def test_slow_and_unfit_variants_and_ties(choose):
    best, ms = choose(TIMES, TIMES, TIMES, fits=[True, True, False, True, True])
    assert best == 4 and ms[2] == np.float32(1e30)
    more = np.where(TIMES > 1.5, 0.1, TIMES)           # beyond 1.5 of the best: not timed again
    best, ms = choose(TIMES, TIMES, more)
    assert best == 2 and ms[0] == np.float32(2.2) and ms[3] == np.float32(1.6)
    assert choose([1.0, 0.99], [1.0, 0.99], [1.0, 0.99])[0] == 0
    assert choose([1.0, 0.98], [1.0, 0.98], [1.0, 0.98])[0] == 1
