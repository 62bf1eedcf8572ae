"""The RHS entry points are as exact as the reference's formulas evaluated in
IEEE 64-bit arithmetic: rms error against extended precision no larger than the
oracle's own in float64, on the same fields."""
import numpy as np
import pytest

from famrdp_jax import cases
from famrdp_jax.core.types import GasModel, Metrics
from famrdp_jax.rhs.invscd import compute_invscd_rhs
from famrdp_jax.rhs.viscous import compute_viscous_rhs
from oracle import numerics as ON

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limiter", ["minmod", "vanleer"])
@pytest.mark.parametrize("metrics", ["unit", "curvilinear"])
@pytest.mark.parametrize("field", ["smooth", "jumps"])
def test_no_larger_error_than_64_bits(field, metrics, limiter):
    print(f"case: {field} {metrics} {limiter}", flush=True)
    rng, shape = np.random.default_rng(41), (24, 21, 28)
    if field == "smooth":
        rho, p = 1 + 0.05 * rng.uniform(-1, 1, shape), 1 + 0.05 * rng.uniform(-1, 1, shape)
        u, v, w = (0.4 + 0.05 * rng.uniform(-1, 1, shape) for _ in range(3))
    else:
        rho, p = np.exp(rng.uniform(-1, 1, shape)), np.exp(rng.uniform(-1, 1, shape))
        u, v, w = (rng.uniform(-2, 2, shape) for _ in range(3))
    q = np.stack([rho, rho * u, rho * v, rho * w, p / 0.4 + 0.5 * rho * (u * u + v * v + w * w)])
    k = np.eye(3)[:, :, None, None, None] + np.zeros((3, 3) + shape)
    vol = np.ones(shape)
    if metrics == "curvilinear":
        k, vol = k + rng.uniform(-0.3, 0.3, (3, 3) + shape), rng.uniform(0.5, 1.5, shape)
    m = Metrics(jac=1.0 / vol, kxyz=k, vol=vol)
    gas = GasModel(gamma=1.4, R=1 / 1.4, mu0=0.02, T0=1.0, Ts=0.383, Pr_lam=0.72)
    got = (compute_invscd_rhs(q, m, ghost=2, gamma=1.4, reconstruct="muscl2", flux="roe", limiter=limiter),
           compute_viscous_rhs(q, m, gas=gas, ghost=2))

    def plain(T):
        x = lambda a: a.astype(T)  # noqa: E731
        gd = {n: T(c) for n, c in cases.gas_dict(gas).items()}
        return (ON.compute_invscd_rhs(x(q), x(k), x(vol), gamma=T(1.4), limiter=limiter),
                ON.compute_viscous_rhs(x(q), x(k), **gd))

    for name, a, b, ref in zip(("inviscid", "viscous"), got, plain(np.float64), plain(np.longdouble)):
        ours, theirs = (float(np.sqrt(((x - ref) ** 2).mean()) / np.abs(ref).max()) for x in (a, b))
        print(f"  {name}: {ours:.3e}, 64 bits {theirs:.3e}", flush=True)
        assert ours <= theirs, name
