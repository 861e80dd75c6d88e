"""Newton-Schulz above 64 states, called again and again on one context: the launch
that finds the convergence stops in every one of its workgroups alike, however many
there are and whatever number of iterations was expected, so that T, the iterations
and the change of T come out the same to the bit each time."""
import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65, 256, 257, 512])
def test_every_call_gives_the_same_bits(gpu, n):
    hmat = np.diag([9.0, 9.0, 9.3]).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / 9.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    with CPContext((27, 27, 30), hmat, ecut, n, *k) as c:
        c.set_psi(psi)
        w, u = np.linalg.eigh(c.overlap() / 2.0)
        c.set_psi((u * np.sqrt(np.linspace(0.5, 1.5, n) / w)) @ u.T @ psi)
        c.overlap()
        first = c.ortho_ns(1e-14, 30)
        assert first[3] and first[1] > 3
        for i in range(8):
            t, it, err, ok = c.ortho_ns(1e-14, 30)  # expects as many as the last call took
            assert ok and (it, err) == first[1:3] and np.array_equal(t, first[0])
            c.ortho_ns(1e-2 if i % 2 else 1e-6, 30)  # ... or fewer
