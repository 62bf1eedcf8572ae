"""The stage kernels' reciprocal and square root (famrdp_math.h rcp, fsqrt) are
rounded once: their last operation adds a correction whose own error is below
2^-70 of the result, so both are within half an ulp and 2^-17 of one."""
import numpy as np
import pytest
import torch

from famrdp_jax import _lib as L

pytestmark = pytest.mark.gpu


def test_reciprocal_and_root_are_rounded_once():
    print("case: fast reciprocal and root of 400000 values", flush=True)
    rng = np.random.default_rng(12)
    x = np.concatenate([np.exp(rng.uniform(-200, 200, 200000)), rng.uniform(0.25, 4.0, 200000)])
    xd = torch.tensor(x, device="cuda")
    r, s = torch.empty_like(xd), torch.empty_like(xd)
    L.check(L.lib().famrdp_fastmath_probe(xd.data_ptr(), r.data_ptr(), s.data_ptr(), None, x.size, L.stream()))
    torch.cuda.synchronize()
    xl = x.astype(np.longdouble)
    for name, got, ref in (("rcp", r, 1 / xl), ("sqrt", s, np.sqrt(xl))):
        ulp = float((np.abs(got.cpu().numpy() - ref) / np.spacing(np.abs(ref).astype(np.float64))).max())
        print(f"  {name}: {ulp:.6f} ulp", flush=True)
        assert ulp <= 0.5 + 2.0 ** -17
