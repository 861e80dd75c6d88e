"""Newton-Schulz iterations beyond those launched one by one run on the whole device
too: a call that expects too few of them takes at most ten times as long as one that
knows the count (one workgroup for all of them took a hundred times as long), and
gives the same bits.  Sizes with one tile per workgroup and with several."""
import time

import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65, 200, 300, 512, 530])
def test_more_iterations_than_expected(gpu, n):
    hmat = np.diag([9.0, 9.0, 9.3]).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / 9.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))

    def call(c, tol):
        t0 = time.perf_counter()
        r = c.ortho_ns(tol, 30)
        return time.perf_counter() - t0, r

    known, late = [], []
    with CPContext((27, 27, 30), hmat, ecut, n, *k) as c:
        c.set_psi(psi)
        w, u = np.linalg.eigh(c.overlap() / 2.0)
        c.set_psi((u * np.sqrt(np.geomspace(0.004, 1.6, n) / w)) @ u.T @ psi)
        c.overlap()
        call(c, 1e-15)
        for _ in range(3):
            s, a = call(c, 1e-15)  # as many as the last call took
            known.append(s)
            few = call(c, 0.9)[1]
            s, b = call(c, 1e-15)  # far more than the last call took
            late.append(s)
            assert a[3] and b[3] and a[1] == b[1] > few[1] + 4
            assert a[2] == b[2] and np.array_equal(a[0], b[0])
    print(f"[n={n}] {few[1]} expected, {a[1]} taken: {min(late) * 1e6:.0f} us, known "
          f"{min(known) * 1e6:.0f} us", flush=True)
    assert min(late) < 10.0 * min(known)
