"""The x passes of the engine with one kernel per axis, which transform row
pairs wave by wave: lengths whose factors lie either way round, odd row counts,
lone last rows, states that do not divide into chunks, planes full of columns.
rho, psi(r) (also after the passes back) and V psi against the Stockham passes in
FP64: 1e-12 of the largest value, and 2e-6 for FP32 transforms (2e-7 in 2-norm,
peaks of a few times that)."""
import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu

GRIDS = [(24, 27, 30), (27, 24, 24), (30, 27, 50), (32, 81, 24), (54, 27, 24), (75, 30, 24),
         (100, 27, 24), (128, 24, 27), (160, 27, 24)]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("grid", GRIDS)
def test_x_passes(gpu, grid, precision):
    nx, ny, nz = grid
    # kx up to nx/3, ky and kz to a quarter: the sphere is an ellipsoid of the box
    hmat = np.diag([nx / 3.0, ny / 4.0, nz / 4.0]).reshape(9)
    ecut = (2.0 * np.pi * 0.97) ** 2
    k = _lib.kvecs(ecut, hmat)
    n = 19
    rng = np.random.default_rng(nx)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    v = rng.normal(size=(nz, ny, nx))

    def run(mode, prec):
        with CPContext(grid, hmat, ecut, n, *k, precision=prec, fft_mode=mode) as c:
            c.set_psi(psi)
            c.set_vks(v)
            c.fft_g2r()
            out = [c.get_density(), c.get_psir(n - 1)]
            c.vpsi_r2g()
            return out + [c.get_force(), c.get_psir(n - 1)]

    a, b = run(3, precision), run(1, "fp64")
    err = [np.abs(x - y).max() / np.abs(y).max() for x, y in zip(a, b)]
    print(grid, precision, ["%.1e" % e for e in err], flush=True)
    assert max(err) < (1e-12 if precision == "fp64" else 2e-6)
