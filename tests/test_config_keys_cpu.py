"""Face-keyed tables of a configuration are found under Face members, plain
ints and anything else that converts to the face's number."""
import numpy as np
import pytest

from famrdp_jax._plan import bcs_from_config, cuts_from_topology
from famrdp_jax.core.constants import BCType, Face
from famrdp_jax.core.types import BlockTopology


@pytest.mark.parametrize("key", [lambda f: f, int, np.int64, lambda f: str(int(f))])
def test_topology_and_parameters_by_any_face_key(key):
    types = [BCType.CUT1TO1, BCType.CUT1TO1, BCType.WALL, BCType.SYMMETRY, BCType.FARFIELD, BCType.OUTFLOW]
    topo = BlockTopology(0, {Face.IMIN: (0, Face.IMAX, 0), Face.IMAX: (0, Face.IMIN, 0)},
                         {key(f): t for f, t in zip(Face, types)})
    params = {key(Face.JMIN): {"wall_type": "isothermal", "T_wall": 2.0}, key(Face.KMIN): {"q_inf": [1, 0, 0, 0, 3]},
              key(Face.KMAX): {"extrapolate": True}}
    assert cuts_from_topology([topo]) == [(0, 0, 0, 1, 0), (0, 1, 0, 0, 0)]
    free = (1.0, 0.0, 0.0, 0.0, 2.5)
    assert bcs_from_config([topo], params) == [
        (0, 2, 1, 2.0, free), (0, 3, 2, 0.0, free), (0, 4, 3, 0.0, (1.0, 0.0, 0.0, 0.0, 3.0)), (0, 5, 4, 0.0, free)]
