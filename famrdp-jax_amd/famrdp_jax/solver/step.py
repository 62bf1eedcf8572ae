"""One TVD-RK3 step on the GPU (famrdp_jax/solver/step.py:18-56)."""
from __future__ import annotations

from .. import _lib as L
from .._plan import plan_for
from ..core.types import Block, Config, State


def step(state: State, cfg: Config, dt: float) -> State:
    """Halo exchange once, BCs once, then three RHS evaluations combined by
    Shu-Osher TVD-RK3 over every padded cell of every block.  Returns a new
    State (t + dt, step + 1); the input arrays are not modified.  With
    ``cfg.nan_check`` (the reference's default) the new state is monitored on
    the GPU and a non-finite or non-positive (rho, p) interior cell raises
    FloatingPointError."""
    src = [L.device_f64(b.q) for b in state.blocks]
    kx = [L.device_f64(m.kxyz) for m in state.metrics]
    vo = [L.device_f64(m.vol) for m in state.metrics]
    dims = [tuple(q.shape[1:]) for q in src]
    plan = plan_for(dims, cfg.topology, cfg.bc_params, cfg.gas, cfg.scheme.limiter, cfg.ghost)
    # several blocks: one launch per stage over all of them instead of one per
    # block (the same bits; 8 blocks of 13^3-44^3 cells, a stage: 112 -> 33 us)
    many = len(src) > 1
    if any(q.requires_grad for q in src) or L.forward_ad():     # autograd, reverse or forward, sees the copy
        qs = [q.clone() for q in src]
        plan.step(qs, kx, vo, dt, batched=many)
    else:
        qs = [L._torch().empty_like(q) for q in src]
        plan.step_from(src, qs, kx, vo, dt, batched=many)
    if cfg.nan_check:
        plan.raise_if_bad(qs)
    blocks = tuple(Block(q=L.like_input(q, b.q), xyz=b.xyz) for q, b in zip(qs, state.blocks))
    return State(blocks=blocks, metrics=state.metrics, t=state.t + dt, step=state.step + 1)
