"""The products of up to 64 states, where a wave holds a whole gram: state counts
at the edges of its 16-tiles and of the next form, in both precisions (FP64
either way: sums of at most 3,000 products, 1e-12 of the largest value).  S is
symmetric to the bit, and Psi T stages only as many rows of T as there are."""
import numpy as np
import pytest

from openatom_amd import _lib, system
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 32, 33, 47, 49, 64])
def test_products(gpu, n, precision):
    hmat = np.diag([9.0, 9.0, 9.3]).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / 9.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi, f = (rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
              for _ in range(2))
    t = rng.normal(size=(n, n))
    with CPContext((27, 27, 30), hmat, ecut, n, *k, precision=precision, gemm_split=3) as c:
        c.set_psi(psi)
        c.set_force(f)
        S, lam = c.overlap(), c.lambda_()
        force = c.get_force()
        c.set_tmat(t)
        c.rotate()
        out = c.get_psi()
    a, b = psi.view(np.float64), f.view(np.float64)
    w = np.repeat(system.gamma_weights(k[0]), 2)
    w = w / w.max() * 2.0
    ref = [(a * w) @ a.T, a @ b.T]
    half = np.repeat(np.where(k[0] == 0, 0.5, 1.0), 2)
    ref += [b - half * (ref[1].T @ a), t.T @ a]
    got = [S, lam, force.view(np.float64), out.view(np.float64)]
    err = [np.abs(x - y).max() / np.abs(y).max() for x, y in zip(got, ref)]
    print(f"[{n} {precision}] " + " ".join(f"{e:.1e}" for e in err), flush=True)
    assert max(err) < 1e-12 and np.array_equal(S, S.T)
