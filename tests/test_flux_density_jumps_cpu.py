"""CPU check of the stage kernels' Roe flux (famrdp_math.h roe_flux2, compiled
for the host) on faces between states of very different density, either side
the lighter one, against flux/roe.py:21-85 in extended precision.

Tolerance: the flux is about 140 operations none of which cancels terms much
larger than the largest flux component, so its error is a few tens of roundings
of that component: 64 of 2^-53.  The reverse is held to
the same number of roundings of what its result depends on: of the largest of
its ten components and of what relative changes of the ten inputs would move it
by (a light side's density cotangent can cancel to far less than its terms)."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest
import torch

from oracle import numerics as ON

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "famrdp-jax_amd", "csrc")
G = 1.4
TOL = 64 * 2.0 ** -53


@pytest.fixture(scope="module")
def hc(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("fhc") / "libfhc.so")
    subprocess.run([hipcc, "--cuda-host-only", "-O1", "-ffp-contract=off", "-std=c++17", "-fPIC", "-shared", "-I" + CSRC,
                    os.path.join(HERE, "hostcheck", "flux_hostcheck.hip"), "-o", out],
                   check=True, capture_output=True)
    return ctypes.CDLL(out)


def faces(ratio, n, seed):
    """States of pressure about 1 and |u| < 0.5, left density `ratio` times the right one, and area vectors."""
    rng = np.random.default_rng(seed)
    side = lambda s: np.stack([s * rng.uniform(0.8, 1.2, n), *(rng.uniform(-0.5, 0.5, n) for _ in range(3)),  # noqa: E731
                               rng.uniform(0.9, 1.1, n)], axis=1)
    return side(min(ratio, 1.0)), side(min(1.0 / ratio, 1.0)), rng.uniform(-1, 1, (n, 3))


RATIOS = [1e-6, 1e-4, 1e-3, 1e-2, 1.0, 1e2, 1e3, 1e4, 1e6]


@pytest.mark.parametrize("full", [0, 1])
@pytest.mark.parametrize("ratio", RATIOS)
def test_flux_between_light_and_heavy(hc, ratio, full):
    n = 500
    pl, pr, S = faces(ratio, n, 31)
    F = np.zeros((n, 5))
    P = lambda a: np.ascontiguousarray(a).ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    hc.hc_roe_flux2(n, full, P(pl), P(pr), P(S), ctypes.c_double(G), P(F))
    x = lambda a: a.T.astype(np.longdouble)  # noqa: E731
    g = np.longdouble(G)
    A = np.sqrt((x(S) ** 2).sum(axis=0))
    ref = (2 * A * ON.roe_flux(ON.prim_to_cons(x(pl), g), ON.prim_to_cons(x(pr), g), x(S) / A, gamma=g)).T
    err = np.abs(F - ref).max(axis=1) / np.abs(ref).max(axis=1)
    print(f"ratio {ratio:g}: max {float(err.max()):.2e}")
    assert float(err.max()) <= TOL


@pytest.mark.parametrize("full", [0, 1])
@pytest.mark.parametrize("speed", [0.1, 0.5, 2.4])
def test_energy_flux_of_equal_states_is_as_exact_as_in_64_bits(hc, speed, full):
    """No waves there: twice (E + p) u.S, rms error no larger than that product's in IEEE arithmetic."""
    n = 20000
    pl, _, S = faces(1.0, n, 91)
    pl[:, 1:4] *= 2 * speed
    F = np.zeros((n, 5))
    P = lambda a: np.ascontiguousarray(a).ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    hc.hc_roe_flux2(n, full, P(pl), P(pl), P(S), ctypes.c_double(G), P(F))

    def plain(T):
        rho, u, v, w, p = pl.T.astype(T)
        s, g = S.T.astype(T), T(G)
        E = p / (g - 1) + rho * (T(0.5) * (u * u + v * v + w * w))
        return 2 * ((E + p) * (u * s[0] + v * s[1] + w * s[2]))

    ref = plain(np.longdouble)
    rms = lambda x: float(np.sqrt(((x - ref) ** 2).mean()))  # noqa: E731
    print(f"speed {speed:g}: {rms(F[:, 4]):.2e}, plain {rms(plain(np.float64)):.2e}")
    assert rms(F[:, 4]) <= rms(plain(np.float64))


@pytest.mark.parametrize("mach", [0.4, 2.0])
def test_rhs_flux_is_as_exact_as_the_formulas_in_64_bits(hc, mach):
    """The RHS entry point's form at equal densities: rms error no larger than that of flux/roe.py in IEEE arithmetic."""
    n = 20000
    pl, pr, S = faces(1.0, n, 91)
    for p in (pl, pr):
        p[:, 1:4] *= 2 * mach * np.sqrt(G * p[:, 4:] / p[:, :1])
    F = np.zeros((n, 5))
    P = lambda a: np.ascontiguousarray(a).ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    hc.hc_roe_flux2(n, 1, P(pl), P(pr), P(S), ctypes.c_double(G), P(F))

    def plain(T):
        x = lambda a: a.T.astype(T)  # noqa: E731
        A, g = np.sqrt((x(S) ** 2).sum(axis=0)), T(G)
        return (2 * A * ON.roe_flux(ON.prim_to_cons(x(pl), g), ON.prim_to_cons(x(pr), g), x(S) / A, gamma=g)).T

    ref = plain(np.longdouble)
    rms = lambda x: np.sqrt((((x - ref) / np.abs(ref).max(axis=1)[:, None]) ** 2).mean(axis=0)).astype(float)  # noqa: E731
    ours, theirs = rms(F), rms(plain(np.float64))
    print(f"mach {mach:g}: {ours}, plain {theirs}")
    assert (ours <= theirs).all()


def _vjp_reference(pl, pr, S, f):
    """Cotangents of flux/roe.py:21-85 times 2 |S|, in extended precision: the complex step through the formulas."""
    g, eps = np.longdouble(G), np.longdouble(1e-30)
    mag = lambda z: np.where(z.real >= 0, z, -z)  # noqa: E731
    out = np.zeros((len(pl), 10), dtype=np.longdouble)
    A = np.sqrt((S.astype(np.longdouble) ** 2).sum(axis=1))
    n = (S / A[:, None]).T
    for k in range(10):
        x = np.concatenate([pl, pr], axis=1).astype(np.clongdouble)
        x[:, k] += 1j * eps
        def conserved(p):
            ke = 0.5 * (p[1] ** 2 + p[2] ** 2 + p[3] ** 2)
            return np.stack([p[0], p[0] * p[1], p[0] * p[2], p[0] * p[3], p[4] / (g - 1) + p[0] * ke])
        L, R = x[:, :5].T, x[:, 5:].T
        UL, UR = conserved(L), conserved(R)
        H = lambda U, p: (U[4] + p[4]) / U[0]  # noqa: E731
        sL, sR = np.sqrt(L[0]), np.sqrt(R[0])
        uh = (sL * L[1:4] + sR * R[1:4]) / (sL + sR)
        Hh = (sL * H(UL, L) + sR * H(UR, R)) / (sL + sR)
        q2 = (uh ** 2).sum(axis=0)
        c2 = (g - 1) * (Hh - 0.5 * q2)
        c, un, rho = np.sqrt(c2), (uh * n).sum(axis=0), sL * sR
        e = np.longdouble("0.1") * (mag(un) + c)
        fix = lambda l: np.where(mag(l).real >= e.real, mag(l), 0.5 * (l * l / e + e))  # noqa: E731
        d = UR - UL
        dp = (g - 1) * (d[4] - (uh * d[1:4]).sum(axis=0) + 0.5 * q2 * d[0])
        dn = (d[1:4] * n).sum(axis=0) - un * d[0]
        a1, a5, a2 = (dp - rho * c * dn) / (2 * c2), (dp + rho * c * dn) / (2 * c2), d[0] - dp / c2
        t = (d[1:4] - uh * d[0]) / rho
        t = t - (t * n).sum(axis=0) * n
        one = np.ones_like(un)
        wave = lambda s: np.stack([one, *(uh + s * c * n), Hh + s * c * un])  # noqa: E731
        shear = np.stack([0 * one, *(rho * t), rho * (uh * t).sum(axis=0)])
        diss = fix(un - c) * a1 * wave(-1) + fix(un + c) * a5 * wave(1) + \
            mag(un) * (a2 * np.stack([one, *uh, 0.5 * q2]) + shear)
        def physical(U, p):
            v = (p[1:4] * n).sum(axis=0)
            return np.stack([U[0] * v, *(U[1:4] * v + p[4] * n), (U[4] + p[4]) * v])
        F = A * (physical(UL, L) + physical(UR, R) - diss)
        out[:, k] = (f.T * F).sum(axis=0).imag / eps
    return out


@pytest.mark.parametrize("ratio", RATIOS)
def test_reverse_between_light_and_heavy(hc, ratio):
    n = 400
    pl, pr, S = faces(ratio, n, 57)
    f = np.random.default_rng(58).uniform(-1, 1, (n, 5))
    lp = np.zeros((2, n, 5))
    P = lambda a: np.ascontiguousarray(a).ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    hc.hc_roe_flux2_vjp(n, P(pl), P(pr), P(S), ctypes.c_double(G), P(f), lp[0].ctypes.data_as(ctypes.c_void_p),
                        lp[1].ctypes.data_as(ctypes.c_void_p))
    ref = _vjp_reference(pl, pr, S, f)
    move = np.zeros(n, dtype=np.longdouble)
    for k in range(10):
        x = np.concatenate([pl, pr], axis=1)
        x[:, k] *= 1 + 1e-6
        move += np.abs(_vjp_reference(x[:, :5], x[:, 5:], S, f) - ref).max(axis=1) / 1e-6
    err = np.abs(np.concatenate([lp[0], lp[1]], axis=1) - ref).max(axis=1) / (np.abs(ref).max(axis=1) + move)
    print(f"ratio {ratio:g}: max {float(err.max()):.2e}")
    assert float(err.max()) <= TOL


@pytest.mark.parametrize("jump", [1.0, 1e-3])
def test_reverse_is_as_exact_as_autograd_in_64_bits(hc, jump):
    """At equal densities, states apart or nearly equal: rms error no larger than autograd's through flux/roe.py."""
    n = 2000
    pl, pr, S = faces(1.0, n, 71)
    pr = pl + jump * (pr - pl)
    f = np.random.default_rng(72).uniform(-1, 1, (n, 5))
    lp = np.zeros((2, n, 5))
    P = lambda a: np.ascontiguousarray(a).ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    hc.hc_roe_flux2_vjp(n, P(pl), P(pr), P(S), ctypes.c_double(G), P(f), lp[0].ctypes.data_as(ctypes.c_void_p),
                        lp[1].ctypes.data_as(ctypes.c_void_p))
    tl, tr, ts = torch.tensor(pl.T, requires_grad=True), torch.tensor(pr.T, requires_grad=True), torch.tensor(S.T)
    A = torch.sqrt((ts ** 2).sum(dim=0))
    F = 2.0 * A * ON.roe_flux(ON.prim_to_cons(tl, G), ON.prim_to_cons(tr, G), ts / A, gamma=G)
    (F * torch.tensor(f.T)).sum().backward()
    ref = _vjp_reference(pl, pr, S, f)
    rms = lambda x: float(np.sqrt((((x - ref) / np.abs(ref).max(axis=1)[:, None]) ** 2).mean()))  # noqa: E731
    ours = rms(np.concatenate([lp[0], lp[1]], axis=1))
    theirs = rms(np.concatenate([tl.grad.numpy().T, tr.grad.numpy().T], axis=1))
    print(f"jump {jump:g}: {ours:.2e}, autograd {theirs:.2e}")
    assert ours <= theirs
