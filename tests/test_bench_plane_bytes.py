"""bench.py's compulsory bytes of the fused plane passes, on the CPU: V counts as the
pass reads it, in its own precision by row class and in FP64 otherwise."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("n,kabs,csz,v", [
    (100, 24, 8, 4), (100, 24, 16, 8),  # by row class
    (100, 25, 8, 8),                    # 4 kmax + 1 > N: not pruned, no row classes
    (90, 22, 8, 8), (90, 22, 16, 8),    # no multiple of 4
])
def test_v_in_the_precision_that_is_read(n, kabs, csz, v):
    geo = dict(nx=n, ny=n, nz=n, nlines=991, nplane_x=kabs + 1, npts=32961, kabs=kabs)
    launch = dict(nchunk=5, pcp=26)
    lines = 2 * 128 * 991 * n * csz
    assert bench.plane_bytes("k_plane_r2g", geo, csz, 128, launch) == lines + 26 * n**3 * v
    assert bench.plane_bytes("k_plane_r2g_rho", geo, csz, 128, launch) \
        == lines + 26 * n**3 * (v + 8)
    assert bench.plane_bytes("k_plane_g2r", geo, csz, 128, launch) == lines // 2 + 5 * n**3 * 8


def test_roofline_of_the_headline_kernel():
    """128 states at 100^3, 26 state chunks, mixed: 307 MB."""
    geo = dict(nx=100, ny=100, nz=100, nlines=991, nplane_x=25, npts=32961, kabs=24)
    res = dict(precision="mixed", geo=geo, launch=dict(nchunk=5, pcp=26),
               timings={"k_plane_r2g": 0.2}, timings_timed={"k_plane_r2g": 0.16})
    r = bench.roofline(res, 128)
    assert r["algorithmic_bytes"] == 306_956_800
    assert r["achieved"] == pytest.approx(306_956_800 / 0.16e-3 / 1e9)
