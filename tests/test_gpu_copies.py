"""Coefficients out of a context: from 8 MiB up they come through a ring of
pinned slots that threads empty.  Every byte comes back, at sizes on both sides
of that line, with ragged last pieces and blocks, into fresh and used buffers at
any 16-byte offset, and nothing beside them is written."""
import ctypes

import numpy as np
import pytest

from openatom_amd import _lib
from openatom_amd.step import CPContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mib", [0.3, 7.9, 8.2, 17.0, 40.3])
def test_get_returns_what_was_set(gpu, mib):
    hmat = np.diag([9.0, 9.0, 9.3]).reshape(9)
    ecut = (2.0 * np.pi * 6.4 / 9.0) ** 2
    k = _lib.kvecs(ecut, hmat)
    n = int(mib * 2**20 / (16 * len(k[0])))
    rng = np.random.default_rng(n)
    psi = rng.normal(size=(n, len(k[0]))) + 1j * rng.normal(size=(n, len(k[0])))
    with CPContext((27, 27, 30), hmat, ecut, n, *k, ns_mode=1) as c:
        c.set_psi(psi)
        assert np.array_equal(c.get_psi(), psi)
        for off in (1, 2, 255):
            buf = np.full(off + psi.size + 3, 7.0 + 7.0j)
            st = c._L.oa_psi_get(c.h, ctypes.c_void_p(buf.ctypes.data + 16 * off))
            assert st == _lib.OA_OK
            assert np.array_equal(buf[off:-3], psi.ravel())
            assert np.all(buf[:off] == 7.0 + 7.0j) and np.all(buf[-3:] == 7.0 + 7.0j)
