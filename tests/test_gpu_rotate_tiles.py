"""Psi T and the Lambda projection above 128 states: the row tiles of a workgroup
follow the state and the point count.  Each of the four pairs (waves x tiles per
wave, on 256 CUs: 4 x 2, 4 x 3, 3 x 3, 4 x 4) with a ragged count of columns and
of rows, against numpy: 1e-12 of the largest value (sums of at most 449
products).  |F| comes from partial sums of the projection, one per workgroup."""
import numpy as np
import pytest

from openatom_amd import _lib, system
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kc,grid", [(257, 9.2, 40), (177, 12.4, 54), (385, 16.0, 64),
                                       (449, 26.4, 108)])
def test_row_tiles(gpu, n, kc, grid):
    side = 20.0
    hmat = np.diag([side] * 3).reshape(9)
    ecut = (2.0 * np.pi * kc / side) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi, f = (rng.normal(size=(n, 2 * len(k[0]))) for _ in range(2))
    t = rng.normal(size=(n, n))
    w = np.repeat(np.where(k[0] == 0, 0.5, 1.0), 2)
    with CPContext((grid, grid, grid), hmat, ecut, n, *k, use_cg=1, dt=0.5) as c:
        c.set_psi(psi.view(np.complex128))
        c.set_force(f.view(np.complex128))
        lam = c.lambda_()
        force = c.get_force().view(np.float64)
        c.set_tmat(t)
        c.rotate()
        out = c.get_psi().view(np.float64)
        red, par = system.redundant_pairs(*k)
        x = psi.copy().view(np.complex128)
        x[:, red] = np.conj(x[:, par])
        x[:, (k[0] == 0) & (k[1] == 0) & (k[2] == 0)] = 1.0
        c.set_psi(x)
        e, u = np.linalg.eigh(c.overlap() / 2.0)
        c.set_psi(((u / np.sqrt(e)) @ u.T @ x.view(np.float64)).view(np.complex128))
        c.set_vks(rng.normal(size=(grid, grid, grid)) * 0.05)
        fnorm = c.step()["fnorm"]
        fstep = c.get_force()
    ref = f - w * (lam.T @ psi)
    err = [np.abs(force - ref).max() / np.abs(ref).max()]
    ref = t.T @ psi
    err.append(np.abs(out - ref).max() / np.abs(ref).max())
    err.append(abs(fnorm - np.linalg.norm(fstep)) / fnorm)
    print(f"[{n} x {psi.shape[1]}] F {err[0]:.1e} Psi T {err[1]:.1e} |F| {err[2]:.1e}", flush=True)
    assert max(err) < 1e-12
