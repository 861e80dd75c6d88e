"""The dense products above 128 states, at the edges of their dispatch.

Psi T and the Lambda projection run in row tiles of 16 (waves x tiles per wave
chosen by the state count: 9 tiles at 144, 12 at 177, 16 at 256, two blocks
above), the split-BF16 Lambda gram in blocks of 128 or 256 rows (256 from 385
to 512 states), with ragged state and point counts.  Checked against numpy on
random coefficients and forces: 1e-12 of the largest value in FP64 (sums of at
most 3,000 products), and 1e-6 for the split gram (operands rounded to FP32,
2^-24 each, FP32 sums over a K slice).  The conjugate-gradient step's |F| comes
from the projection's own partial sums, and its update writes the redundant
kx = 0 points from their partners."""
import numpy as np
import pytest

from openatom_amd import _lib, system
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu

STATES = (129, 144, 177, 193, 256, 300, 390, 513)


def build(n):
    hmat = np.diag([9.0, 9.0, 9.3]).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / 9.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    x = [rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0]))) for _ in range(2)]
    return dict(grid=(27, 27, 30), hmat=hmat, ecut=ecut, k=k, psi=x[0], f=x[1],
                t=rng.normal(size=(n, n)))


def reals(a):
    return np.ascontiguousarray(a).view(np.float64)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", STATES)
def test_products(gpu, n, precision):
    s = build(n)
    with CPContext(s["grid"], s["hmat"], s["ecut"], n, *s["k"], precision=precision) as c:
        c.set_psi(s["psi"])
        c.set_force(s["f"])
        lam = c.lambda_()
        f = c.get_force()
        c.set_tmat(s["t"])
        c.rotate()
        psi = c.get_psi()
    a, b = reals(s["psi"]), reals(s["f"])
    ref = a @ b.T
    tol = 1e-12 if precision == "fp64" else 1e-6
    w = np.where(s["k"][0] == 0, 0.5, 1.0)
    fref = s["f"] - w * (lam.T @ a).view(np.complex128)
    pref = (s["t"].T @ a).view(np.complex128)
    err = [np.abs(lam - ref).max() / np.abs(ref).max(), np.abs(f - fref).max() / np.abs(fref).max(),
           np.abs(psi - pref).max() / np.abs(pref).max()]
    print(f"[{n} {precision}] Lambda {err[0]:.1e} F {err[1]:.1e} Psi T {err[2]:.1e}", flush=True)
    assert err[0] < tol and err[1] < 1e-12 and err[2] < 1e-12


@pytest.mark.parametrize("n", [5, 129, 300])
def test_cg_norm_and_redundant_points(gpu, n):
    s = build(n)
    kx, ky, kz = s["k"]
    red, par = system.redundant_pairs(kx, ky, kz)
    psi = system.initial_coeffs(kx, ky, kz, s["hmat"], n, 3)
    v = np.random.default_rng(1).normal(size=s["grid"][::-1])
    with CPContext(s["grid"], s["hmat"], s["ecut"], n, kx, ky, kz, use_cg=1, dt=1.0) as c:
        c.set_psi(psi)
        c.set_vks(v)
        r = [c.step() for _ in range(2)][-1]
        f, p = c.get_force(), c.get_psi()
    assert abs(r["fnorm"] - np.linalg.norm(f)) < 1e-12 * r["fnorm"]
    assert np.abs(p[:, red] - np.conj(p[:, par])).max() < 1e-12 * np.abs(p).max()
