"""The RHS entry points on states a caller looks for: the non-finite values are
the oracle's exactly (jnp.maximum floors of flux/roe.py:23-39, minmod and van
Leer of physics/reconstruct/muscl2.py:5-12, Sutherland's power), the others
agree to the existing bar of the RHS parity tests, over the largest finite value
of each variable."""
import numpy as np
import pytest

from famrdp_jax import cases
from famrdp_jax.core.types import GasModel, Metrics
from famrdp_jax.rhs.invscd import compute_invscd_rhs
from famrdp_jax.rhs.viscous import compute_viscous_rhs
from oracle import numerics as ON

pytestmark = pytest.mark.gpu
TOL = 1e-12
BAD = {"density -0.5": (0, -0.5), "density 0": (0, 0.0), "density nan": (0, np.nan), "density inf": (0, np.inf),
       "momentum nan": (2, np.nan), "momentum inf": (1, np.inf), "energy inf": (4, np.inf), "energy -inf": (4, -np.inf),
       "energy nan": (4, np.nan), "no pressure": (4, -0.3), "area 0": None}


def _same(name, got, ref):
    # (an energy can be infinite where the oracle's is NaN: a contracted product
    # does not overflow before the sum that takes it)
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref), err_msg=name)
    for v in range(5):
        ok = np.isfinite(ref[v])
        if ok.any():
            assert np.abs(got[v][ok] - ref[v][ok]).max() <= TOL * max(np.abs(ref[v][ok]).max(), 1.0), (name, v)


@pytest.mark.parametrize("limiter", ["minmod", "vanleer"])
@pytest.mark.parametrize("bad", BAD)
def test_non_finite_values_are_the_oracles(bad, limiter):
    print(f"case: {bad} {limiter}", flush=True)
    rng, shape = np.random.default_rng(19), (9, 11, 10)
    rho, p = rng.uniform(0.8, 1.2, shape), rng.uniform(0.8, 1.2, shape)
    u, v, w = (rng.uniform(-0.5, 0.5, shape) for _ in range(3))
    q = np.stack([rho, rho * u, rho * v, rho * w, p / 0.4 + 0.5 * rho * (u * u + v * v + w * w)])
    k = np.eye(3)[:, :, None, None, None] + rng.uniform(-0.2, 0.2, (3, 3) + shape)
    vol = rng.uniform(0.5, 1.5, shape)
    if BAD[bad] is None:
        k[:, :, 4, 5, :] = 0.0
        k[:, :, 5, 5, :] = 0.0
    else:
        for cell in ((4, 5, 4), (7, 3, 7)):
            q[(BAD[bad][0],) + cell] = BAD[bad][1]
    m = Metrics(jac=1.0 / vol, kxyz=k, vol=vol)
    gas = GasModel(gamma=1.4, R=1 / 1.4, mu0=0.02, T0=1.0, Ts=0.383, Pr_lam=0.72)
    with np.errstate(all="ignore"):
        inv = ON.compute_invscd_rhs(q, k, vol, gamma=1.4, limiter=limiter)
        vis = ON.compute_viscous_rhs(q, k, **cases.gas_dict(gas))
    _same("inviscid", compute_invscd_rhs(q, m, ghost=2, gamma=1.4, reconstruct="muscl2", flux="roe", limiter=limiter), inv)
    _same("viscous", compute_viscous_rhs(q, m, gas=gas, ghost=2), vis)
