"""Newton-Schulz on an S whose eigenvalues lie far apart (ratios of 25, 100 and 1000)
in every form (ns_mode): T against (S/2)^{-1/2} by
eigendecomposition.  A product over n terms is off by about sqrt(n) eps of its
largest, and the iteration hands an error on by no more than the ratio of the
eigenvalues; four times that leaves room for the products of the last iterations.
X' = C X / 2 in place of X C / 2 (C = 3I - T X) multiplies rounding errors by up to
half the square root of the ratio in every iteration and fails from a ratio of 50."""
import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def inv_sqrt(s):
    w, u = np.linalg.eigh(s)
    return (u / np.sqrt(w)) @ u.T


@pytest.mark.parametrize("mode,n", [(m, n) for m in range(7) for n in (40, 128, 300)
                                    if not (m == 5 and n == 40)])  # row blocks in four parts
def test_context(gpu, mode, n):
    hmat = np.diag([9.0, 9.0, 9.3]).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / 9.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    u, _ = np.linalg.qr(rng.standard_normal((n, n)))
    with CPContext((27, 27, 30), hmat, ecut, n, *k, ns_mode=mode) as c:
        c.set_psi(psi)
        psi = inv_sqrt(c.overlap() / 2.0) @ psi
        for ratio in (25.0, 100.0, 1000.0):
            c.set_psi((u * np.sqrt(np.geomspace(1.6 / ratio, 1.6, n))) @ u.T @ psi)
            s = c.overlap()
            t, it, rms, ok = c.ortho_ns(1e-15, 30)
            ref = inv_sqrt(s / 2.0)
            err = np.abs(t - ref).max() / np.abs(ref).max()
            print(f"[ns_mode {mode}, n={n}, ratio {ratio:g}] {it} iterations, {err:.1e}",
                  flush=True)
            assert ok and err < 4.0 * np.sqrt(n) * ratio * EPS


@pytest.mark.parametrize("n", [16, 48, 100, 270])
def test_stateless(gpu, n):
    """Ten iterations at most: a ratio of 25 takes all of them."""
    rng = np.random.default_rng(n)
    u, _ = np.linalg.qr(rng.standard_normal((n, n)))
    s = 2.0 * (u * np.geomspace(1.6 / 25.0, 1.6, n)) @ u.T
    t, _ = _lib.ortho_transform(s)
    ref = inv_sqrt(s / 2.0)
    err = np.abs(t - ref).max() / np.abs(ref).max()
    print(f"[n={n}] {err:.1e}", flush=True)
    assert err < 4.0 * np.sqrt(n) * 25.0 * EPS
