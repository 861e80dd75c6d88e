"""V_KS by the two-factor passes on every axis: lengths whose factors lie either
way round, odd row counts, lone last rows, ragged last workgroups.  Without ions
V_KS = V_xc + V_Hartree: against numpy on the context's own density, 1e-11 of the
largest value (the transforms' rounding is 1e-15, the Hartree factor's spread of
4 pi/G^2 some hundreds), the energies to 1e-11."""
import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu

GRIDS = [(24, 27, 30), (27, 24, 50), (75, 30, 24), (100, 27, 24), (54, 81, 24), (24, 24, 160),
         (24, 150, 27), (144, 24, 36)]


def pz(r):
    c = np.cbrt(r)
    rs = 0.62035049089940001667 / c
    xf = -0.98474502184269654118 * c
    s, l = np.sqrt(rs), np.log(rs)
    c1 = 1.0 + 1.0529 * s + 0.3334 * rs
    c2 = 1.0 + 7.0 / 6.0 * 1.0529 * s + 4.0 / 3.0 * 0.3334 * rs
    lo = 0.0311 * l - 0.048 + 0.002 * rs * l - 0.0116 * rs
    ml = (0.0311 * l + (-0.048 - 0.0311 / 3.0) + 2.0 / 3.0 * 0.002 * rs * l
          + (2.0 * -0.0116 - 0.002) * rs / 3.0)
    cf = np.where(rs >= 1.0, -0.1423 / c1, lo)
    mf = np.where(rs >= 1.0, -0.1423 / c1 * c2 / c1, ml)
    return xf, cf, xf + mf


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("grid", GRIDS)
def test_v_of_rho(gpu, grid, precision):
    nx, ny, nz = grid
    a = np.array(grid) / 4.2  # |k| up to a fifth of each length, twice that in rho
    hmat = np.diag(a).reshape(9)
    ecut = (2.0 * np.pi * 0.97) ** 2
    k = _lib.kvecs(ecut, hmat)
    n = 5
    rng = np.random.default_rng(nx)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    with CPContext(grid, hmat, ecut, n, *k, precision=precision, vks_from_rho=1) as c:
        c.set_psi(psi)
        c.fft_g2r()
        rho, v, r = c.get_density(), c.get_vks(), c.result()
    vol, pts = a.prod(), nx * ny * nz
    f = [np.fft.fftfreq(m, 1.0 / m) * 2.0 * np.pi / b for m, b in zip((nz, ny, nx), a[::-1])]
    g2 = f[0][:, None, None] ** 2 + f[1][None, :, None] ** 2 + f[2][None, None, :] ** 2
    g = np.fft.fftn(rho) * vol / pts
    on = (g2 > 0) & (g2 <= 4.0 * ecut)
    hf = np.where(on, 4.0 * np.pi / (np.where(on, g2, 1.0) * vol), 0.0)
    xf, cf, vxc = pz(rho)
    ref = vxc + np.fft.ifftn(hf * g).real * pts
    eh = 0.5 * (hf * np.abs(g) ** 2).sum()
    exc = ((0.75 * xf + cf) * rho).sum() * vol / pts
    err = [np.abs(v - ref).max() / np.abs(ref).max(), abs(r["ehart"] / eh - 1.0),
           abs(r["exc"] / exc - 1.0)]
    print(grid, precision, ["%.1e" % e for e in err], flush=True)
    assert max(err) < 1e-11
