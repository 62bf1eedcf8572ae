"""The RHS entry points at tile edges and remainders, against the oracle, and
on blocks that no face updates whatever their volumes hold.  Tolerance: the
existing bar of the RHS parity tests."""
import numpy as np
import pytest
import torch

from famrdp_jax import cases
from famrdp_jax.core.types import GasModel, Metrics
from famrdp_jax.rhs.invscd import compute_invscd_rhs
from famrdp_jax.rhs.viscous import compute_viscous_rhs
from oracle import numerics as ON

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _case(shape, seed):
    rng = np.random.default_rng(seed)
    rho, p = rng.uniform(0.8, 1.2, shape), rng.uniform(0.8, 1.2, shape)
    u, v, w = (rng.uniform(-0.5, 0.5, shape) for _ in range(3))
    q = np.stack([rho, rho * u, rho * v, rho * w, p / 0.4 + 0.5 * rho * (u * u + v * v + w * w)])
    k = np.eye(3)[:, :, None, None, None] + rng.uniform(-0.2, 0.2, (3, 3) + shape)
    vol = rng.uniform(0.5, 1.5, shape)
    return q, Metrics(jac=1.0 / vol, kxyz=k, vol=vol)


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 5), (4, 4, 8), (5, 9, 17), (8, 8, 16), (18, 19, 33), (6, 41, 20),
                                   (33, 5, 18)])
@pytest.mark.parametrize("limiter", ["minmod", "vanleer"])
def test_rhs_terms_at_tile_edges(shape, limiter):
    print(f"case: {shape} {limiter}", flush=True)
    q, m = _case(shape, 11)
    got = compute_invscd_rhs(q, m, ghost=2, gamma=1.4, reconstruct="muscl2", flux="roe", limiter=limiter)
    ref = ON.compute_invscd_rhs(q, m.kxyz, m.vol, gamma=1.4, limiter=limiter)
    assert np.abs(got - ref).max() <= TOL * max(np.abs(ref).max(), 1.0)
    gas = GasModel(gamma=1.4, R=1 / 1.4, mu0=0.02, T0=1.0, Ts=0.383, Pr_lam=0.72)
    got = compute_viscous_rhs(q, m, gas=gas, ghost=2)
    ref = ON.compute_viscous_rhs(q, m.kxyz, **cases.gas_dict(gas))
    assert np.abs(got - ref).max() <= TOL * max(np.abs(ref).max(), 1.0)


def test_cells_no_axis_updates_are_zero_whatever_the_volume():
    q, m = _case((4, 4, 4), 3)
    for vol in (0.0, np.inf, np.nan):
        mm = Metrics(jac=m.jac, kxyz=m.kxyz, vol=np.full((4, 4, 4), vol))
        got = compute_invscd_rhs(q, mm, ghost=2, gamma=1.4, reconstruct="muscl2", flux="roe", limiter="minmod")
        assert not got.any() and not np.signbit(got).any()
