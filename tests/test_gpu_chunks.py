"""State chunks of a G->R pass whose workgroups have a whole plane and a CU to themselves
(150 points in FP64): a rho partial weighs little beside such a workgroup's states, so
the chunks are as many as fill the rounds of workgroups (three were 9 % slower at 80
states).  The density keeps its sum rule."""
import numpy as np
import pytest

from openatom_amd import _lib, system
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nst,chunks", [(16, 3), (80, 5)])
def test_whole_planes_with_a_cu_each(gpu, nst, chunks):
    n, side = 150, 10.0
    hmat = np.diag([side, side, side]).reshape(9)
    ecut = (2.0 * np.pi * 37.3 / side) ** 2  # as many columns as the pruned passes take
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(nst)
    psi = rng.normal(size=(nst, len(k[0]))) + 1j * rng.normal(size=(nst, len(k[0])))
    red, par = system.redundant_pairs(*k)
    psi[:, red] = np.conj(psi[:, par])
    psi[:, (k[0] == 0) & (k[1] == 0) & (k[2] == 0)] = 1.0
    with CPContext((n, n, n), hmat, ecut, nst, *k) as c:
        assert c.config["engine"] in (3, 4) and c.config["nchunk"] == chunks
        c.set_psi(psi)
        c.set_vks(np.zeros((n, n, n)))
        c.fft_g2r()
        rho = c.get_density()
    norm = ((np.abs(psi) ** 2) * system.gamma_weights(k[0])).sum()
    assert abs(rho.sum() * side ** 3 / n ** 3 - norm) < 1e-12 * norm
