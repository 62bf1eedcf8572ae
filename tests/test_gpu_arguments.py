"""Arguments that a plan refuses, and what the plan does after it has."""
import pytest
import torch

from famrdp_jax import cases
from famrdp_jax._plan import plan_for
from _util import to_dev

pytestmark = pytest.mark.gpu


def _two_blocks():
    state, cfg = cases.case_c3(nb_axis=2, lo=9, hi=14)[:2]
    state = to_dev(state)
    plan = plan_for([tuple(b.q.shape[1:]) for b in state.blocks], cfg.topology, cfg.bc_params, cfg.gas,
                    cfg.scheme.limiter, cfg.ghost)
    return plan, [b.q for b in state.blocks], [m.kxyz for m in state.metrics], [m.vol for m in state.metrics]


def test_step_from_refuses_arrays_that_share_memory():
    """A permutation of the input arrays as output, and an output that begins inside another block's input."""
    print("case: step_from into arrays that overlap its input", flush=True)
    plan, src, kx, vo = _two_blocks()
    into = [torch.empty_like(q) for q in src]
    plan.step_from(src, into, kx, vo, 1e-3)
    want = [q.clone() for q in into]
    same = max(range(1, len(src)), key=lambda b: src[b].numel())
    for swap in (src[same], src[same].reshape(-1)[-1:]):
        bad = list(into)
        bad[0] = swap
        with pytest.raises(ValueError, match="shares memory"):
            plan.step_from(src, bad, kx, vo, 1e-3)
    plan.step_from(src, into, kx, vo, 1e-3)
    for q, w in zip(into, want):
        assert torch.equal(q, w)
