"""Newton-Schulz by plain launches: one workgroup up to 64 states, tiles of 16
up to 256, of 32 above, at the edges of the tiles, the 64-deep batches and the
three forms.  T against (S/2)^{-1/2} by
eigendecomposition: S/2 has eigenvalues within a factor of five of each other,
so a few n eps of both sides stay below 1e-11 of the largest value.  Where
fewer iterations were launched than convergence takes, the last launch runs
the others by the same arithmetic: T is the same to the bit."""
import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


def inv_sqrt(s):
    w, u = np.linalg.eigh(s)
    return (u / np.sqrt(w)) @ u.T


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 48, 49, 63, 64, 65, 79, 128, 129, 255,
                               256, 257, 271, 272, 321])
def test_edges(gpu, n):
    rng = np.random.default_rng(n)
    u, _ = np.linalg.qr(rng.standard_normal((n, n)))
    s = 2.0 * (u * np.linspace(0.4, 1.6, n)) @ u.T
    T, st = _lib.ortho_transform(s)
    ref = inv_sqrt(s / 2.0)
    err = np.abs(T - ref).max() / np.abs(ref).max()
    print(f"[n={n}] {st} {err:.1e}", flush=True)
    assert st == _lib.OA_OK and err < 1e-11


@pytest.mark.parametrize("n", [65, 130, 272])
def test_iterations_past_the_expected_count(gpu, n):
    hmat = np.diag([9.0, 9.0, 9.3]).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / 9.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    u, _ = np.linalg.qr(rng.standard_normal((n, n)))
    mix = (u * np.sqrt(np.linspace(0.2, 1.6, n))) @ u.T

    def one(first_tol):
        with CPContext((27, 27, 30), hmat, ecut, n, *k, ns_mode=6) as c:
            c.set_psi(psi)
            c.set_psi(mix @ inv_sqrt(c.overlap() / 2.0) @ psi)
            s = c.overlap()
            if first_tol:
                c.ortho_ns(first_tol, 30)
            t, it, err, ok = c.ortho_ns(1e-15, 30)
        return s, t, it, ok

    s, t, it, ok = one(None)
    s2, t2, it2, ok2 = one(0.5)  # its two or three iterations are what the second call expects
    err = np.abs(t - inv_sqrt(s / 2.0)).max() / np.abs(t).max()
    print(f"[n={n}] iterations {it}, {it2} err {err:.1e}", flush=True)
    assert ok and ok2 and it == it2 and it > 5
    assert np.array_equal(s, s2) and np.array_equal(t, t2)
    assert err < 1e-11


@pytest.mark.parametrize("n", [40, 65, 272])
def test_a_value_that_is_not_finite_is_reported(gpu, n):
    """Also with more iterations allowed than are launched: no convergence, T lost."""
    hmat = np.diag([9.0, 9.0, 9.3]).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / 9.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    psi[n // 2, 7] = np.nan
    with CPContext((27, 27, 30), hmat, ecut, n, *k, ns_mode=6) as c:
        c.set_psi(psi)
        c.overlap()
        t, it, err, ok = c.ortho_ns(1e-15, 30)
    assert not ok and it == 30 and np.isnan(err) and np.isnan(t).all()
