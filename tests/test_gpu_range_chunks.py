"""State ranges are cut into chunks of their own: uneven ranges down to one state, at
lengths of the three kinds of plane passes.  As for the chunks of all states, the
density is that of one call up to the order of the chunk sums (1e-13, sums in FP64)
and the forces are the same to the bit."""
import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,nst", [(27, 64), (54, 40), (75, 48), (150, 12)])
def test_uneven_ranges(gpu, n, nst, precision):
    side = 10.0
    hmat = np.diag([side] * 3).reshape(9)
    ecut = (2.0 * np.pi * ((n - 1) // 4 + 0.3) / side) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(nst, len(k[0]))) + 1j * rng.normal(size=(nst, len(k[0])))
    with CPContext((n, n, n), hmat, ecut, nst, *k, precision=precision) as c:
        assert c.config["engine"] in (3, 4)
        c.set_psi(psi)
        c.set_vks(rng.normal(size=(n, n, n)))
        c.fft_g2r()
        rho = c.get_density()
        eke = c.vpsi_r2g()
        force = c.get_force()
        edges = [0, 1, 3, nst // 2, nst - 1, nst]
        ranges = [(a, b - a) for a, b in zip(edges, edges[1:])]
        for s0, ns in ranges:
            c.fft_g2r_states(s0, ns, first=s0 == 0)
        err = np.abs(c.get_density() - rho).max() / np.abs(rho).max()
        part = sum(c.vpsi_r2g_states(s0, ns) for s0, ns in ranges)
        same = np.array_equal(c.get_force(), force)
    print(f"[{n} {nst} {precision}] rho {err:.1e} EKE {abs(part - eke) / eke:.1e}", flush=True)
    assert err < 1e-13 and same and abs(part - eke) < 1e-13 * eke
