"""Reading coefficients behind a queue of steps: the threads that empty the pinned ring
start when the copy can, so the wait costs the process no more than its one caller and
what the runtime itself polls (four threads polling took 4 to 5 CPU seconds a second)."""
import time

import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


def test_waiting_for_queued_steps(gpu):
    n = 400  # 31 MB of coefficients: four threads
    hmat = np.diag([18.0, 18.0, 18.0]).reshape(9)
    ecut = (2.0 * np.pi * 13.2 / 18.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    rng = np.random.default_rng(5)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    with CPContext((54, 54, 54), hmat, ecut, n, *k, want_resid=0) as c:
        c.set_psi(psi)
        w, u = np.linalg.eigh(c.overlap() / 2.0)
        c.set_psi((u / np.sqrt(w)) @ u.T @ psi)
        c.set_vks(np.zeros((54, 54, 54)))
        c.step()
        c.get_psi()  # the ring is there
        time.sleep(0.5)  # numpy's own threads stop polling
        for _ in range(150):
            c.step(fetch=False)
        cpu, wall = time.process_time(), time.perf_counter()
        out = c.get_psi()
        cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
    print(f"{wall * 1e3:.0f} ms, {cpu / wall:.2f} CPUs", flush=True)
    assert np.isfinite(out).all() and wall > 0.05
    assert cpu < 2.5 * wall
