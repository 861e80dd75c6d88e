"""Projections of few atoms onto more than 64 states, at the edges of the column
tiles and of the 64-row blocks.  A state's projections do not depend on the other
states: the same rows in a context of 40 states, whose products the oracle's tests
cover, give the same numbers to 1e-13 of the largest (another order of 3,000 sums)."""
import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,atoms", [(65, 1), (70, 15), (128, 16), (129, 17), (96, 32), (70, 33)])
def test_rows_are_independent(gpu, n, atoms):
    hmat = np.diag([9.0, 9.0, 9.3]).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / 9.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    pos = rng.uniform(0.0, 9.0, (atoms, 3))
    grid = np.arange(200) * 0.05
    proj = np.zeros((1, 4, 200))
    proj[0, 0] = np.exp(-0.3 * grid ** 2)

    def z(rows):
        with CPContext((27, 27, 30), hmat, ecut, len(rows), *k, ns_mode=1) as c:
            c.set_nonlocal(pos, np.zeros(atoms, np.int32), 0.0, 0.05, proj, np.ones(1), np.ones(1))
            c.set_psi(rows)
            return c.nonlocal_get()[0]

    big, small = z(psi), z(psi[-40:])
    err = np.abs(big[-40:] - small).max() / np.abs(small).max()
    print(f"[{n} states, {atoms} atoms] {err:.1e}", flush=True)
    assert np.isfinite(big).all() and err < 1e-13
