"""Plane passes by row class (oa_plane4.h) at every length that has classes.

The pruned transforms of the lengths that are multiples of 4 run by row class;
fft_full = 1 runs the plane passes over whole planes instead.  Only the order
of the additions differs, so density, forces and kinetic energy agree to
rounding: 1e-13 relative in FP64, 1e-6 in mixed precision (the bars of the
pruned against the full transforms).  The sphere reaches |k| = (N - 1) / 4, the
largest the pruned passes take, or stays two columns below it; the z axis has a
length of its own, the state count is no multiple of a chunk, and occupations
differ.  One more step with fixed V runs the R->G pass that also sums rho where
it is compiled."""
import numpy as np
import pytest

from openatom_amd import system
from openatom_amd.step import CPContext
from tests.helpers import rel

pytestmark = pytest.mark.gpu

SIZES = (24, 32, 36, 40, 48, 60, 64, 72, 80, 96, 100, 108, 120, 128, 144, 160)
NST = 5


def build(n, below):
    kmax = (n - 1) // 4 - below
    nz = 24 if n != 24 else 27
    side = 9.0
    # along z the sphere must fit the shorter grid: |kz| <= (nz - 1) / 4
    sz = side * ((nz - 1) // 4 + 0.3) / (kmax + 0.3)
    hmat = np.diag([side, side, sz]).reshape(9)
    ecut = (2.0 * np.pi * (kmax + 0.3) / side) ** 2
    from openatom_amd import _lib
    kx, ky, kz = _lib.kvecs(ecut, hmat)
    assert max(np.abs(kx).max(), np.abs(ky).max()) == kmax
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(NST, len(kx))) + 1j * rng.normal(size=(NST, len(kx)))
    red, par = system.redundant_pairs(kx, ky, kz)
    psi[:, red] = np.conj(psi[:, par])
    psi[:, (kx == 0) & (ky == 0) & (kz == 0)] = 1.0
    return dict(grid=(n, n, nz), hmat=hmat, ecut=ecut, k=(kx, ky, kz), psi=psi,
                v=rng.normal(size=(nz, n, n)), occ=np.array([1.0, 0.75, 1.0, 0.5, 0.25]))


def run(s, precision, full, keep=0):
    with CPContext(s["grid"], s["hmat"], s["ecut"], NST, *s["k"], occ=s["occ"],
                   precision=precision, fft_full=full, psir_keep=keep, use_lambda=0, dt=1e-3,
                   ns_tol=1e300) as c:
        c.set_psi(s["psi"])
        c.set_vks(s["v"])
        c.fft_g2r()
        rho, psir = c.get_density(), c.get_psir(NST - 1)
        eke = c.vpsi_r2g()
        f = c.get_force()
        c.step()
        return dict(rho=rho, psir=psir, f=f, eke=np.array([eke]), rho_step=c.get_density(),
                    f_step=c.get_force(), engine=c.config["engine"])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", SIZES)
def test_row_classes_equal_whole_planes(gpu, n, precision):
    s = build(n, 2 if n % 3 == 0 else 0)
    a, b = run(s, precision, 0), run(s, precision, 1)
    same = 1e-13 if precision == "fp64" else 1e-6
    assert a["engine"] in (3, 4)
    err = {k: rel(a[k], b[k]) for k in a if k != "engine"}
    print(f"[{n} {precision}]", {k: f"{v:.1e}" for k, v in err.items()}, flush=True)
    assert all(v < same for v in err.values()), err
    # the density's sum rule: sum rho = sum_s occ_s <psi_s|psi_s> N / Omega
    w = system.gamma_weights(s["k"][0])
    norm = ((np.abs(s["psi"]) ** 2) * w).sum(axis=1)
    expect = (s["occ"] * norm).sum() * a["rho"].size / abs(np.linalg.det(s["hmat"].reshape(3, 3)))
    assert abs(a["rho"].sum() - expect) < 10 * same * expect
