"""Contacts of large density ratio, the lighter side on either side of the face
along each axis: the inviscid RHS entry point and a whole step against the
oracle.  Tolerance: the existing bar of the RHS and step parity tests."""
import numpy as np
import pytest
import torch

from famrdp_jax.core.types import Block, BlockTopology, Config, GasModel, Metrics, SchemeChoice, State
from famrdp_jax.rhs.invscd import compute_invscd_rhs
from famrdp_jax.solver.stepper import Stepper
from oracle import blocks as OB
from oracle import numerics as ON
from _util import rel_linf, to_dev

pytestmark = pytest.mark.gpu
TOL = 1e-12
SHAPE = (12, 13, 18)


def contact(axis, ratio, seed):
    """Two uniform streams that meet at the middle of the axis, p about 1, |u| < 0.5, the first one's density `ratio`
    times smaller than the other's (larger for ratio < 1); random metrics.  (Uniform, so that the largest term is the
    contact's and not some acoustic noise of the light side.)"""
    rng = np.random.default_rng(seed)
    idx = np.arange(SHAPE[axis]).reshape([-1 if a == axis else 1 for a in range(3)])
    first = np.broadcast_to(idx < SHAPE[axis] // 2, SHAPE)
    x = [np.where(first, a, b) for a, b in ((min(1 / ratio, 1.0), min(ratio, 1.0)), (1.0, 1.05), (0.3, -0.1), (-0.2, 0.2),
                                            (0.1, 0.4))]
    rho, p, u, v, w = x
    q = np.stack([rho, rho * u, rho * v, rho * w, p / 0.4 + 0.5 * rho * (u * u + v * v + w * w)])
    k = np.eye(3)[:, :, None, None, None] + rng.uniform(-0.2, 0.2, (3, 3) + SHAPE)
    vol = rng.uniform(0.5, 1.5, SHAPE)
    return q, Metrics(jac=1.0 / vol, kxyz=k, vol=vol)


@pytest.mark.parametrize("limiter", ["minmod", "vanleer"])
@pytest.mark.parametrize("ratio", [1e2, 1e-2, 1e4, 1e-4, 1e6, 1e-6])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_contact(axis, ratio, limiter):
    print(f"case: contact of {ratio:g} along axis {axis}, {limiter}", flush=True)
    q, m = contact(axis, ratio, 17 + axis)
    x = lambda a: a.astype(np.longdouble)  # noqa: E731
    ref = ON.compute_invscd_rhs(x(q), x(m.kxyz), x(m.vol), gamma=np.longdouble(1.4), limiter=limiter)
    got = compute_invscd_rhs(q, m, ghost=2, gamma=1.4, reconstruct="muscl2", flux="roe", limiter=limiter)
    err = float(np.abs(got - ref).max() / np.abs(ref).max())
    print(f"  rhs {err:.2e}", flush=True)
    assert err <= TOL
    # a step of a quarter of the light side's acoustic limit, without viscosity
    gas = GasModel(gamma=1.4, R=1 / 1.4, mu0=0.0, T0=1.0, Ts=0.383, Pr_lam=0.72)
    dt = 0.25 * 0.5 / (3 * 1.4 * np.sqrt(1.4 * 1.05 / min(ratio, 1 / ratio)))
    topo = BlockTopology(0, {}, {})
    cfg = Config(gas=gas, scheme=SchemeChoice("muscl2", "roe", 3, limiter), bc_params={}, topology=(topo,), ghost=2,
                 nan_check=False)
    gd = dict(gamma=1.4, R=1 / 1.4, mu0=0.0, T0=1.0, Ts=0.383, Pr_lam=0.72)
    want = OB.step([q], [(m.kxyz, m.vol)], [topo], {}, gd, dt, limiter=limiter)[0]
    assert np.isfinite(want).all()
    state = State(blocks=(Block(q=q, xyz=np.zeros(1)),), metrics=(m,))
    for tile in (None, 1, 6, 12, 18, 20):       # by size, then fused, split, re-staging, marching and wide
        st = Stepper(to_dev(state), cfg)
        if tile is not None:
            st.plan.set_tile(tile)
        st.advance(dt)
        torch.cuda.synchronize()
        err = rel_linf(st.qs[0].cpu().numpy(), want)
        print(f"  step, variant {tile}: {err:.2e}", flush=True)
        assert err <= TOL
