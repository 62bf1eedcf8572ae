"""Arguments that a plan refuses, and what the plan does after it has."""
import pytest
import torch

from famrdp_jax import _lib as L
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


def test_a_refused_call_leaves_the_plan_bound_as_it_was():
    """A call with a NULL state after a valid one, then a valid one with the other pointers of the refused call."""
    print("case: NULL state pointer between two steps", flush=True)
    plan, src, kx, vo = _two_blocks()
    first, second = [q.clone() for q in src], [q.clone() for q in src]
    plan.step(first, kx, vo, 1e-3, batched=True)
    second[1:] = first[1:]                       # the second call differs in block 0 alone
    rest = [q.clone() for q in second]
    ptrs = plan._ptrs(second)
    ptrs[len(src) - 1] = None
    rc = plan._lib.famrdp_step(plan._h, ptrs, plan._ptrs(kx), plan._ptrs(vo), 1e-3, 1, L.stream())
    with pytest.raises(ValueError, match="is NULL"):
        L.check(rc)
    keep = first[0].clone()
    plan.step(second, kx, vo, 1e-3, batched=True)
    plan.step(rest, kx, vo, 1e-3, batched=True)
    assert torch.equal(first[0], keep)
    for q, w in zip(second, rest):
        assert torch.equal(q, w)


def test_replays_of_a_captured_step_between_in_place_ones():
    """A functional step in a graph and a resident stepper of one configuration share a plan: each replay writes the
    plan's block table, and the stepper's next step must not run on it."""
    from famrdp_jax.solver.step import step
    from famrdp_jax.solver.stepper import Stepper
    print("case: captured functional step and in-place steps in turn", flush=True)
    state, cfg = cases.case_c3(nb_axis=2, lo=9, hi=14)[:2]
    state, dt = to_dev(state), 1e-3
    ref = Stepper(state, cfg)
    ref.advance(dt, 4, batched=True)
    want, once = [q.clone() for q in ref.qs], [b.q for b in step(state, cfg, dt).blocks]
    st = Stepper(state, cfg)
    st.advance(dt, 1, batched=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(state, cfg, dt)
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = step(state, cfg, dt)
    for _ in range(3):
        st.advance(dt, 1, batched=True)
        for b in out.blocks:
            b.q.zero_()
        g.replay()
        torch.cuda.synchronize()
        for b, w in zip(out.blocks, once):
            assert torch.equal(b.q, w)
    for q, w in zip(st.qs, want):
        assert torch.equal(q, w)


def test_forward_mode_sees_the_copy_as_reverse_mode_does():
    from famrdp_jax.core.types import Block, State
    from famrdp_jax.solver.step import step
    from torch.autograd import forward_ad as fwd
    print("case: functional step of dual tensors", flush=True)
    state, cfg = cases.case_c3(nb_axis=2, lo=9, hi=14)[:2]
    state = to_dev(state)
    plain = [b.q for b in step(state, cfg, 1e-3).blocks]
    tangents = [torch.rand_like(b.q) for b in state.blocks]
    with fwd.dual_level():
        dual = State(blocks=tuple(Block(q=fwd.make_dual(b.q.clone(), t), xyz=b.xyz)
                                  for b, t in zip(state.blocks, tangents)), metrics=state.metrics)
        for b, t, q in zip(step(dual, cfg, 1e-3).blocks, tangents, plain):
            primal, tangent = fwd.unpack_dual(b.q)
            assert torch.equal(primal, q) and torch.equal(tangent, t)


def test_state_check_under_another_default_device():
    from dataclasses import replace
    from famrdp_jax.solver.step import step
    from famrdp_jax.solver.stepper import Stepper
    print("case: nan_check with torch's default device set to the GPU", flush=True)
    state, cfg = cases.case_c1(9)[:2]
    state, cfg = to_dev(state), replace(cfg, nan_check=True)
    torch.set_default_device("cuda")
    try:
        out = step(state, cfg, 1e-3)
        st = Stepper(state, cfg)
        st.advance(1e-3, 1)
    finally:
        torch.set_default_device(None)
    assert torch.equal(out.blocks[0].q, st.qs[0])
