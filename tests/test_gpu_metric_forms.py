"""Grid metrics of both forms -- a thread per cell, and marched in tiles -- on
grids either side of the line between them, against the oracle.  Tolerance and
random grids as for the tiles' edges."""
import numpy as np
import pytest

from famrdp_jax.mesh.metric import compute_metrics
from oracle import metric as OM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    (260, 16, 70), (171, 48, 36), (2100, 5, 31), (33, 130, 64), (9, 200, 150), (65, 64, 64), (33, 64, 64),   # marched
    (63, 64, 65), (31, 64, 64), (300, 300, 5), (400, 230, 3), (3, 300, 9), (171, 47, 34), (30, 9, 1000)])    # by cells
def test_metrics_of_both_forms(shape):
    print(f"case: {shape}", flush=True)
    rng = np.random.default_rng(8)
    grid = np.stack(np.meshgrid(*(np.arange(n, dtype=np.float64) for n in shape), indexing="ij"))
    xyz = grid + rng.uniform(-0.1, 0.1, (3,) + shape)
    m = compute_metrics(xyz, ghost=2)
    jac, kxyz, vol = OM.compute_metrics(xyz)[:3]
    assert np.array_equal(m.vol, np.abs(m.jac))
    assert np.abs(m.jac - jac).max() <= 1e-11 * max(np.abs(jac).max(), 1.0)
    safe = np.abs(jac) > 0.2
    assert safe.mean() > 0.2
    assert np.abs((m.kxyz - kxyz)[:, :, safe]).max() <= 1e-11 * np.abs(kxyz[:, :, safe]).max()
