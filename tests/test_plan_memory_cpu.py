"""A plan whose host tables do not fit in memory is refused with an error; the
exception does not leave the C entry (which would end the process)."""
import os
import subprocess
import sys

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "famrdp-jax_amd")
CODE = """
import ctypes, resource
from famrdp_jax import _lib as L
lib = L.load()
n = 3_000_000
dims = (L.i32 * (3 * n))(*([4] * (3 * n)))
size = int([l for l in open("/proc/self/status") if l.startswith("VmSize")][0].split()[1]) * 1024
resource.setrlimit(resource.RLIMIT_AS, (size + (150 << 20), size + (150 << 20)))
out, gas = L.vp(), L.Gas(1.4, 1.0, 0.0, 1.0, 0.4, 0.7)
print("rc", lib.famrdp_plan_create(ctypes.byref(out), n, dims, 0, None, 0, None, ctypes.byref(gas), 0, 2, 1), flush=True)
print("handle", out.value, lib.famrdp_last_error().decode(), flush=True)
"""


def test_out_of_host_memory_is_an_error():
    res = subprocess.run([sys.executable, "-c", CODE], capture_output=True, text=True, timeout=300,
                         env=dict(os.environ, PYTHONPATH=PKG))
    assert res.returncode == 0, (res.returncode, res.stderr[-500:])
    assert "rc -2" in res.stdout and "handle None" in res.stdout and "host memory" in res.stdout, res.stdout
