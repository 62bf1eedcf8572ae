"""The functional step against the in-place one, bit for bit: block counts on
both sides of one launch's share of the block table, odd block sizes, an input
that only 8-byte loads can read, and an input that autograd follows."""
import pytest
import torch

from famrdp_jax import cases
from famrdp_jax.core.types import Block, State
from famrdp_jax.solver.step import step
from famrdp_jax.solver.stepper import Stepper
from _util import to_dev

pytestmark = pytest.mark.gpu


def _state(nblocks):
    if nblocks == 1:
        state, cfg = cases.case_c1(9)[:2]
    else:
        state, cfg = cases.case_c3(nb_axis=nblocks, lo=9, hi=14)[:2]
    return to_dev(state), cfg


@pytest.mark.parametrize("axis_blocks", [1, 2, 3])
@pytest.mark.parametrize("form", ["plain", "misaligned", "grad"])
def test_functional_step_same_bits_as_in_place(axis_blocks, form):
    state, cfg = _state(axis_blocks)
    print(f"case: {len(state.blocks)} blocks, {form}", flush=True)
    dt = 1e-3
    st = Stepper(state, cfg)
    st.advance(dt, 1)
    qs = []
    for b in state.blocks:
        q = b.q.clone()
        if form == "misaligned":
            flat = torch.empty(q.numel() + 1, dtype=q.dtype, device=q.device)
            flat[1:] = q.reshape(-1)
            q = flat[1:].view(q.shape)
            assert q.data_ptr() % 16 == 8
        elif form == "grad":
            q.requires_grad_(True)
        qs.append(q)
    inp = State(blocks=tuple(Block(q=q, xyz=b.xyz) for q, b in zip(qs, state.blocks)), metrics=state.metrics)
    before = [q.detach().clone() for q in qs]
    out = step(inp, cfg, dt)
    for q, q0, o, ref in zip(qs, before, out.blocks, st.qs):
        assert torch.equal(q.detach(), q0)
        assert o.q.data_ptr() != q.data_ptr() and o.q.requires_grad == (form == "grad")
        assert torch.equal(o.q.detach(), ref)
