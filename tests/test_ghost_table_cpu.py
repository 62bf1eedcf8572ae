"""CPU check of the ghost table (famrdp_ghost.h): exchange and boundary
conditions of a step resolved into one table, against the oracle's halo
exchange followed by its boundary conditions face by face (mesh/halo.py:56-92,
physics/bc/dispatch.py:11-32), for random topologies -- glued blocks, periodic
axes, every kind of boundary on every face, blocks down to the smallest, whose
mirror layers are the opposite ghost layers -- with the entries of a launch in
either order."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from famrdp_jax._plan import bcs_from_config, cuts_from_topology
from famrdp_jax.core.constants import BCType, Face
from famrdp_jax.core.types import BlockTopology
from oracle import blocks as OB

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "famrdp-jax_amd", "csrc")
PAIR = {Face.IMIN: Face.IMAX, Face.IMAX: Face.IMIN, Face.JMIN: Face.JMAX, Face.JMAX: Face.JMIN, Face.KMIN: Face.KMAX,
        Face.KMAX: Face.KMIN}
GAMMA, R = 1.4, 1.0 / 1.4


@pytest.fixture(scope="module")
def hc(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("ghc") / "libghc.so")
    subprocess.run([hipcc, "--cuda-host-only", "-O1", "-ffp-contract=off", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                    os.path.join(HERE, "hostcheck", "ghost_hostcheck.hip"), "-o", out],
                   check=True, capture_output=True)
    return ctypes.CDLL(out)


def _case(seed):
    rng = np.random.default_rng(seed)
    nb = int(rng.integers(1, 4))
    dims = [tuple(int(n) for n in rng.integers(4, 9, 3)) for _ in range(nb)]
    if nb > 1:
        dims[1] = tuple(rng.permutation(dims[0]).tolist()) if rng.random() < 0.3 else dims[0]
    topos = []
    params = {f: {"q_inf": np.array([1.0, 0.3, 0.1, -0.2, 2.6]) + 0.1 * int(f), "extrapolate": bool(rng.random() < 0.7),
                  "wall_type": "isothermal" if rng.random() < 0.5 else "adiabatic", "T_wall": 0.9 + 0.1 * int(f)}
              for f in Face}
    for b in range(nb):
        nbrs, kinds = {}, {}
        for f in Face:
            ax = int(f) // 2
            other = int(rng.integers(0, nb))
            tang = [dims[b][a] for a in range(3) if a != ax]
            if rng.random() < 0.45 and [dims[other][a] for a in range(3) if a != ax] == tang:
                nbrs[f], kinds[f] = (other, PAIR[f] if rng.random() < 0.8 else f, 0), BCType.CUT1TO1
            else:
                nbrs[f] = None
                kinds[f] = rng.choice([BCType.WALL, BCType.SYMMETRY, BCType.FARFIELD, BCType.OUTFLOW])
        topos.append(BlockTopology(b, nbrs, kinds))
    qs = []
    for d in dims:
        rho = rng.uniform(0.6, 1.4, d)
        m = rng.uniform(-0.5, 0.5, (3,) + d)
        qs.append(np.concatenate([rho[None], m, (rng.uniform(1.5, 2.5, d) + 0.5 * (m ** 2).sum(0) / rho)[None]]))
    return dims, topos, params, qs


@pytest.mark.parametrize("reverse", [0, 1])
def test_table_equals_exchange_then_faces(hc, reverse):
    seen = np.zeros(3, dtype=int)
    for seed in range(150):
        dims, topos, params, qs = _case(seed)
        want = [OB.apply_bc(q, t, params, GAMMA, R, 2) for q, t in zip(OB.halo_exchange(qs, topos, 2), topos)]
        cuts = np.array([c[:4] for c in cuts_from_topology(topos)], dtype=np.int32).reshape(-1, 4)
        bcs = bcs_from_config(topos, params)
        ib = np.array([b[:3] for b in bcs], dtype=np.int32).reshape(-1, 3)
        tw = np.array([b[3] for b in bcs], dtype=np.float64)
        qi = np.array([b[4] for b in bcs], dtype=np.float64).reshape(-1, 5)
        d = np.array(dims, dtype=np.int32)
        got = [q.copy() for q in qs]
        ptrs = (ctypes.c_void_p * len(got))(*[g.ctypes.data for g in got])
        n = np.zeros(3, dtype=np.int32)
        P = lambda a: a.ctypes.data_as(ctypes.c_void_p)
        hc.ghost_apply(len(dims), P(d), len(cuts), P(cuts), len(bcs), P(ib), P(tw), P(qi), ctypes.c_double(GAMMA),
                       ctypes.c_double(R), reverse, ptrs, P(n))
        seen += n > 0
        for g, w in zip(got, want):
            np.testing.assert_allclose(g, w, rtol=1e-13, atol=1e-13, err_msg=f"seed {seed}")
    assert (seen > 0).all()      # every part of the table was in use
