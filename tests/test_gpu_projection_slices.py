"""K slices of the projections: Z and Z with its derivatives have a count of their own,
bounded by the buffer of the largest atom set.  Atom sets that grow and shrink in one
context, at the edges of the dispatch (32 and 33 states, 32 and 33 columns), against
NumPy: Z from the table's sums to 1e-12 of the largest value (sums of 1,100 products),
the forces on the ions against a context of their own to the same."""
import numpy as np
import pytest

from openatom_amd import _lib, system
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 32, 33, 64, 65, 130])
def test_atom_sets_of_one_context(gpu, n):
    side = 9.0
    hmat = np.diag([side] * 3).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / side) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    proj = np.zeros((1, 4, 200))
    proj[0, 0] = 1.0  # a projector that is the same at every |G|
    pos = rng.uniform(0.0, side, (40, 3))
    g = 2.0 * np.pi / side * np.array(k, dtype=np.float64)
    w = system.gamma_weights(k[0])

    def make():
        return CPContext((27, 27, 27), hmat, ecut, n, *k)

    def get(c, na):
        c.set_nonlocal(pos[:na], np.zeros(na, np.int32), 0.0, 0.05, proj, np.ones(1), np.ones(1))
        z, e, f = c.nonlocal_get(True)
        assert np.abs(z - c.nonlocal_get()[0]).max() < 1e-12 * np.abs(z).max()
        return z, e, f

    with make() as c:
        c.set_psi(psi)
        for na in (8, 1, 33, 9, 32, 40, 2):
            z, e, f = get(c, na)
            ref = ((psi * w) @ np.exp(1j * g.T @ pos[:na].T)).real / np.sqrt(4.0 * np.pi)
            err = np.abs(z - ref).max() / np.abs(ref).max()
            with make() as d:
                d.set_psi(psi)
                z2, e2, f2 = get(d, na)
            err2 = max(np.abs(z - z2).max() / np.abs(z2).max(), abs(e - e2) / abs(e2),
                       np.abs(f - f2).max() / np.abs(f2).max())
            print(f"[{n} states, {na} atoms] {err:.1e} {err2:.1e}", flush=True)
            assert err < 1e-12 and err2 < 1e-12
