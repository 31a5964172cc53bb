"""The tridiagonal sweep of the projection at the level counts where it changes:
one group of 16 levels more or less, a partial last group, and the longest
column that stays in LDS (64 levels in FP64) and the first that does not.
Against the oracle, 1e-12 normwise as for every pressure test.
"""
import pytest

from tests._golden import interior, normwise
from tests.test_gpu_fft_sizes import TOL, _gpu_pres, _oracle_pres

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ktot", [6, 15, 16, 17, 33, 64, 65])
def test_sweep_group_edges(ktot):
    from tests.golden.make_golden import make_inputs
    p, i = make_inputs(dict(itot=18, jtot=15, ktot=ktot, stretch=True, anelastic=True, dx=50.0, dy=40.0, growth=1.02,
                            seed=ktot))
    out, uvw = _gpu_pres(p, i, 0.37, generic=False)
    d, ref = _oracle_pres(p, i, uvw, 0.37)
    m = interior(d)
    for name in ("ut", "vt", "wt"):
        err = normwise(out[name], ref[name], m)
        assert err < TOL, f"{name}: {err:.3e}"
    err = normwise(out["p"][d.kstart - 1:d.kend], ref["p"][d.kstart - 1:d.kend])
    assert err < TOL, f"p: {err:.3e}"
