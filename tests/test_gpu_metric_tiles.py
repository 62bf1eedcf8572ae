"""Grid metrics at tile and segment edges against the oracle (random grids:
every difference, wrap and column matters).  Tolerance: 1e-11 of each array's
largest value times the condition of the random Jacobians, bounded by keeping
their determinants away from zero."""
import numpy as np
import pytest

from famrdp_jax.mesh.metric import compute_metrics
from oracle import metric as OM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 5, 7), (5, 8, 32), (6, 9, 33), (17, 7, 31), (20, 16, 70), (70, 41, 100),
                                   (100, 9, 35)])
def test_metrics_at_tile_and_segment_edges(shape):
    print(f"case: {shape}", flush=True)
    rng = np.random.default_rng(5)
    grid = np.stack(np.meshgrid(*(np.arange(n, dtype=np.float64) for n in shape), indexing="ij"))
    xyz = grid + rng.uniform(-0.1, 0.1, (3,) + shape)
    m = compute_metrics(xyz, ghost=2)
    jac, kxyz, vol = OM.compute_metrics(xyz)[:3]
    safe = np.abs(jac) > 0.2
    assert safe.mean() > 0.2
    assert np.abs(m.jac - jac).max() <= 1e-11 * np.abs(jac).max()
    assert np.array_equal(m.vol, np.abs(m.jac))
    assert np.abs((m.kxyz - kxyz)[:, :, safe]).max() <= 1e-11 * np.abs(kxyz[:, :, safe]).max()


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 2, 2), (1, 9, 40)])
def test_metrics_of_degenerate_blocks(shape):
    print(f"case: {shape}", flush=True)
    xyz = np.random.default_rng(6).uniform(0.0, 1.0, (3,) + shape)
    m = compute_metrics(xyz, ghost=2)
    # a difference along 1 or 2 cells is zero but for its three roundings, of
    # values up to 8: 3 * 8 * 2^-53 / 12 < 3e-16; the other entries of the
    # Jacobian are below 18 / 12, and the determinant has six terms
    assert np.abs(m.jac).max() <= 6 * 3e-16 * 1.5 ** 2
    assert np.array_equal(m.vol, np.abs(m.jac))
