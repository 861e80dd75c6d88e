"""psi(r) kept between the plane passes (psir_keep = 1, V from rho so that the passes run
separately) at every compiled length: the R->G pass reads what the G->R pass has stored,
by row class (four classes at 160 points in FP64) or in whole planes.  The same density
and V to the bit, and forces and kinetic energy equal to rounding with psi(r)
recomputed: 1e-13 relative in FP64, 1e-6 in mixed precision."""
import numpy as np
import pytest

from openatom_amd.step import CPContext
from tests.helpers import rel
from tests.test_gpu_rowclass import NST, SIZES, build

WHOLE = (27, 30, 45, 50, 54, 75, 81, 90, 150)

pytestmark = pytest.mark.gpu


def run(s, precision, keep):
    with CPContext(s["grid"], s["hmat"], s["ecut"], NST, *s["k"], occ=s["occ"],
                   precision=precision, psir_keep=keep, vks_from_rho=1) as c:
        assert c.config["engine"] == 3
        c.set_psi(s["psi"])
        c.fft_g2r()
        rho, v = c.get_density(), c.get_vks()
        eke = c.vpsi_r2g()
        f = c.get_force()
        psir = c.get_psir(NST - 1)
    return rho, v, f, eke, psir


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", SIZES + WHOLE)
def test_kept_equals_recomputed(gpu, n, precision):
    s = build(n, 2 if n % 3 == 0 else 0)
    a, b = run(s, precision, 1), run(s, precision, 0)
    same = 1e-13 if precision == "fp64" else 1e-6
    print(f"[{n} {precision}] F {rel(a[2], b[2]):.1e} eke {abs(a[3] - b[3]):.1e} psi(r) "
          f"{rel(a[4], b[4]):.1e}", flush=True)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    assert rel(a[2], b[2]) < same and abs(a[3] - b[3]) <= same * abs(b[3])
    assert rel(a[4], b[4]) < same
