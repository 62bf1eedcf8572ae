"""The wide stage kernel and the choice of a stage kernel by size, against the
fused kernel's first shape: bit for bit, in plain and batched launches."""
import pytest
import torch

from famrdp_jax._plan import Plan
from famrdp_jax.core.types import GasModel

pytestmark = pytest.mark.gpu


def _arrays(dims, seed):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *n: torch.rand(n, dtype=torch.float64, generator=g)
    qs, ks, vs = [], [], []
    for d in dims:
        q = torch.stack([torch.ones(d), *(torch.full(d, 0.1) for _ in range(3)), torch.full(d, 2.5)]).double()
        qs.append((q * (1.0 + 0.05 * rnd(5, *d))).cuda())
        ks.append((torch.eye(3).double().reshape(3, 3, 1, 1, 1) + 0.1 * rnd(3, 3, *d)).contiguous().cuda())
        vs.append((1.0 + 0.1 * rnd(*d)).cuda())
    return qs, ks, vs


def _steps(plan, dims, seed, batched):
    qs, ks, vs = _arrays(dims, seed)
    for _ in range(2):
        plan.step(qs, ks, vs, 0.05, batched=batched)
    return qs


GAS = GasModel(R=1 / 1.4, mu0=1e-2, T0=1.0, Ts=0.4)


# smallest blocks (modulo wrap), tile remainders along each axis, both wrap
# forms, tiles inside the block, several blocks
@pytest.mark.parametrize("limiter", ["minmod", "vanleer"])
@pytest.mark.parametrize("dims", [[(4, 4, 4)], [(5, 7, 9)], [(17, 18, 19)], [(23, 37, 41)], [(6, 5, 70)],
                                  [(21, 24, 24), (4, 30, 11), (19, 18, 25)]])
def test_wide_variants_same_bits(dims, limiter):
    print(f"case: {dims} {limiter}", flush=True)
    plan = Plan(dims, [], [], GAS, limiter)
    plan.set_tile(0)
    ref = _steps(plan, dims, 7, False)
    assert all(torch.isfinite(r).all() for r in ref)
    for v in (19, 20):
        plan.set_tile(v)
        for batched in (False, True):
            for a, r in zip(_steps(plan, dims, 7, batched), ref):
                assert torch.equal(a, r), (v, batched)


# sizes on both sides of each line of the choice
@pytest.mark.parametrize("dims,want", [([(20, 20, 20)], 19), ([(36, 36, 36)], 19), ([(32, 32, 32)], 20),
                                       ([(60, 60, 60)], 1), ([(80, 80, 80)], 12), ([(132, 132, 132)], 18),
                                       ([(20, 20, 20)] * 4, 19), ([(52, 52, 52)] * 2, 12)])
def test_untuned_plan_chooses_by_size(dims, want):
    print(f"case: {dims}", flush=True)
    plan = Plan(dims, [], [], GAS, "minmod")
    assert plan.tile()[0] == want
    got = {batched: _steps(plan, dims, 3, batched) for batched in (False, True)}
    plan.set_tile(0)
    ref = _steps(plan, dims, 3, True)
    for batched in (False, True):
        for a, r in zip(got[batched], ref):
            assert torch.equal(a, r)
