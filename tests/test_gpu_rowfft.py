"""Transforms by lane groups (FP64 and the mixed mode) at the lengths where their
plan changes: one to four passes, every radix, rows that do not fill a group, odd
numbers of rows (a pair with one row), 8 to 64 lanes per row (few and many rows),
the wide instance (864, 1000), and a length without a plan (686).  Against the
oracle: FP64 1e-12 normwise as for every pressure test; mixed 1e-5 up to 512
points, the bound of the FP32 transforms in test_gpu_fft_sizes.py, and in proportion
to the length above: p is rounded by eps |p|, and against the gradient of its
largest wave, 2 pi |p| / (n dx), the difference of two neighbours is off by a
relative eps n / (2 pi) (2e-5 at 2048 points).
"""
import pytest

from tests._golden import interior, normwise
from tests.test_gpu_fft_sizes import TOL, _gpu_pres, _oracle_pres

pytestmark = pytest.mark.gpu

SIZES = [(4, 6, 6), (13, 11, 6), (33, 16, 7), (75, 90, 9), (77, 26, 6), (96, 50, 6), (250, 36, 6), (360, 21, 6),
         (864, 8, 6), (12, 1000, 6), (960, 12, 6), (10, 1024, 6), (20, 686, 6), (32, 24, 160)]


def _case(itot, jtot, ktot):
    from tests.golden.make_golden import make_inputs
    return make_inputs(dict(itot=itot, jtot=jtot, ktot=ktot, stretch=True, anelastic=True, dx=50.0, dy=40.0,
                            growth=1.01, seed=itot + 3 * jtot))


@pytest.mark.parametrize("itot,jtot,ktot", SIZES)
def test_fp64(itot, jtot, ktot):
    p, i = _case(itot, jtot, ktot)
    out, uvw = _gpu_pres(p, i, 0.37, generic=True)
    d, ref = _oracle_pres(p, i, uvw, 0.37)
    m = interior(d)
    for name in ("ut", "vt", "wt"):
        err = normwise(out[name], ref[name], m)
        assert err < TOL, f"{name}: {err:.3e}"
    err = normwise(out["p"][d.kstart - 1:d.kend], ref["p"][d.kstart - 1:d.kend])
    assert err < TOL, f"p: {err:.3e}"


@pytest.mark.parametrize("itot,jtot,ktot", [(13, 11, 6), (75, 90, 9), (250, 36, 6), (864, 8, 6), (10, 960, 6),
                                            (2048, 6, 6)])
def test_mixed(itot, jtot, ktot):
    from microhh_amd import abi
    p, i = _case(itot, jtot, ktot)
    out, uvw = _gpu_pres(p, i, 0.37, generic=True, precision=abi.MHH_MIXED)
    d, ref = _oracle_pres(p, i, uvw, 0.37)
    m = interior(d)
    for name in ("ut", "vt", "wt"):
        err = normwise(out[name], ref[name], m)
        assert err < 1e-5 * max(1.0, max(itot, jtot) / 512.0), f"{name}: {err:.3e}"
