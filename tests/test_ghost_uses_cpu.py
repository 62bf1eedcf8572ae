"""CPU check of the ghost table's other two uses (famrdp_ghost.h) on the random
topologies of the table's own check: a step from one set of arrays into another,
and the inner layers of isothermal walls recorded for the reverse sweep, each as
the faces before it have left it (physics/bc/dispatch.py:11-32)."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from famrdp_jax._plan import BC_WALL_ISOTHERMAL, bcs_from_config, cuts_from_topology
from famrdp_jax.core.constants import Face
from famrdp_jax.core.types import BlockTopology
from oracle import blocks as OB
from test_ghost_table_cpu import CSRC, GAMMA, HERE, R, _case


@pytest.fixture(scope="module")
def hc(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("guhc") / "libguhc.so")
    subprocess.run([hipcc, "--cuda-host-only", "-O1", "-ffp-contract=off", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                    os.path.join(HERE, "hostcheck", "ghost_uses_hostcheck.hip"), "-o", out],
                   check=True, capture_output=True)
    return ctypes.CDLL(out)


def P(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _pointers(arrays):
    return (ctypes.c_void_p * len(arrays))(*[a.ctypes.data for a in arrays])


def _arguments(dims, topos, params):
    """The configuration as the host check takes it, and its boundary conditions."""
    cuts = np.array([c[:4] for c in cuts_from_topology(topos)], dtype=np.int32).reshape(-1, 4)
    bcs = bcs_from_config(topos, params)
    ib = np.array([b[:3] for b in bcs], dtype=np.int32).reshape(-1, 3)
    tw = np.array([b[3] for b in bcs], dtype=np.float64)
    qi = np.array([b[4] for b in bcs], dtype=np.float64).reshape(-1, 5)
    d = np.array(dims, dtype=np.int32)
    keep = (d, cuts, ib, tw, qi)
    return (len(dims), P(d), len(cuts), P(cuts), len(bcs), P(ib), P(tw), P(qi), ctypes.c_double(GAMMA), ctypes.c_double(R)), \
        bcs, keep


@pytest.mark.parametrize("reverse", [0, 1])
def test_from_one_set_of_arrays_into_another(hc, reverse):
    kept = 0
    for seed in range(150):
        dims, topos, params, qs = _case(seed)
        want = [OB.apply_bc(q, t, params, GAMMA, R, 2) for q, t in zip(OB.halo_exchange(qs, topos, 2), topos)]
        args, _, keep = _arguments(dims, topos, params)
        out = []
        for q in qs:
            o = np.full_like(q, np.nan)
            o[:, 2:-2, 2:-2, 2:-2] = q[:, 2:-2, 2:-2, 2:-2]
            out.append(o)
        before = [q.copy() for q in qs]
        kept += hc.ghost_out(*args, reverse, _pointers(qs), _pointers(out))
        for q, b, o, w in zip(qs, before, out, want):
            np.testing.assert_array_equal(q, b)
            np.testing.assert_allclose(o, w, rtol=1e-13, atol=1e-13, err_msg=f"seed {seed}")
    assert kept > 0


@pytest.mark.parametrize("reverse", [0, 1])
def test_records_of_isothermal_walls(hc, reverse):
    late = walls = 0
    for seed in range(150):
        dims, topos, params, qs = _case(seed)
        args, bcs, keep = _arguments(dims, topos, params)
        maxc, count = np.zeros(6, dtype=np.int64), [0] * 6
        for b, f, *_ in bcs:
            n = [dims[b][a] for a in range(3) if a != f // 2]
            maxc[f], count[f] = max(maxc[f], n[0] * n[1]), count[f] + 1
        snap = [np.full((max(count[f], 1), 2, 5, max(int(maxc[f]), 1)), np.nan) for f in range(6)]
        want = [s.copy() for s in snap]
        cur, at = OB.halo_exchange(qs, topos, 2), [0] * 6
        for b, (q, t) in enumerate(zip(cur, topos)):      # every face on the result of the ones before
            for f in Face:
                kind = [x[2] for x in bcs if x[0] == b and x[1] == int(f)]
                if not kind:
                    continue
                if kind[0] == BC_WALL_ISOTHERMAL:
                    e, ax, n = [x[0] for x in bcs if x[1] == int(f)].index(b), int(f) // 2, q.shape[1 + int(f) // 2]
                    for gl in range(2):
                        inner = 3 - gl if int(f) % 2 == 0 else n - 4 + gl
                        layer = np.take(q, inner, axis=1 + ax).reshape(5, -1)
                        want[int(f)][e, gl, :, :layer.shape[1]] = layer
                    walls += 1
                only = BlockTopology(t.block_id, {}, {f: t.bc_type[f]})
                q = OB.apply_bc(q, only, params, GAMMA, R, 2)
        got = [q.copy() for q in qs]
        late += hc.ghost_snaps(*args, reverse, _pointers(got), P(maxc), _pointers(snap))
        for f in range(6):
            np.testing.assert_allclose(snap[f], want[f], rtol=1e-13, atol=1e-13, err_msg=f"seed {seed} face {f}")
    assert late > 0 and walls > 100
