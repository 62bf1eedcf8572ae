"""Functional steps of blocks with faces that nothing writes (no condition, plain
outflow or inflow): their ghost cells keep the input's values, and the step is
the in-place one's bit for bit."""
import pytest
import torch

from famrdp_jax import cases
from famrdp_jax.core.constants import BCType, Face
from famrdp_jax.core.types import BlockTopology, Config, State
from famrdp_jax.solver.step import step
from famrdp_jax.solver.stepper import Stepper
from _util import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kinds", [{}, {Face.IMIN: BCType.OUTFLOW, Face.KMAX: BCType.INFLOW},
                                   {Face.JMIN: BCType.WALL, Face.JMAX: BCType.OUTFLOW, Face.IMAX: BCType.SYMMETRY}])
@pytest.mark.parametrize("blocks", [1, 17])
def test_faces_that_nothing_writes(kinds, blocks):
    print(f"case: {blocks} blocks, {kinds}", flush=True)
    state, cfg = cases.case_c1(9)[:2]
    state = to_dev(State(blocks=state.blocks * blocks, metrics=state.metrics * blocks))
    cfg = Config(gas=cfg.gas, scheme=cfg.scheme, bc_params={}, topology=tuple(BlockTopology(b, {}, kinds)
                                                                             for b in range(blocks)), ghost=2,
                 nan_check=False)
    before = [b.q.clone() for b in state.blocks]
    out = step(state, cfg, 1e-3)
    st = Stepper(state, cfg)
    st.advance(1e-3, 1)
    for b, q0, o, ref in zip(state.blocks, before, out.blocks, st.qs):
        assert torch.equal(b.q, q0) and torch.equal(o.q, ref)
