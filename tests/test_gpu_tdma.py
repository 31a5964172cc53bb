"""The tridiagonal sweep of the projection at the level counts where it changes:
one group of 16 levels more or less, a partial last group, and the longest
column that stays in LDS (64 levels of an FP64 spectrum, 128 of an FP32 one) and the first
that does not.  The mixed mode sweeps an FP32 spectrum in FP64 and leaves out
the mean mode.

Against the oracle, tendencies and (not in the mixed mode, whose p is without the
mean profile) p.  FP64: 1e-12 normwise as for every pressure test.  Mixed: 1e-5, the bound
of the FP32 transforms.  FP32: the column of the mean mode, which plain FP32 sweeps
along, has the condition number |A| |A^-1| = 4 K (K + 1) / 2 in the largest norm (a
second difference with a gradient condition below and a value above), about 2 K^2 for K
levels: 2 K^2 2^-24, and not less than the 1e-5 of the transforms.
"""
import pytest

from tests._golden import interior, normwise
from tests.test_gpu_fft_sizes import TOL, _gpu_pres, _oracle_pres

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ktot,precision", [(k, "fp64") for k in (6, 15, 16, 17, 33, 64, 65)]
                         + [(k, q) for q in ("mixed", "fp32") for k in (15, 16, 17, 128, 129)])
def test_sweep_group_edges(ktot, precision):
    from microhh_amd import abi
    from tests.golden.make_golden import make_inputs
    p, i = make_inputs(dict(itot=18, jtot=15, ktot=ktot, stretch=True, anelastic=True, dx=50.0, dy=40.0, growth=1.02,
                            seed=ktot))
    out, uvw = _gpu_pres(p, i, 0.37, generic=False,
                         precision=dict(fp64=abi.MHH_FP64, fp32=abi.MHH_FP32, mixed=abi.MHH_MIXED)[precision])
    d, ref = _oracle_pres(p, i, uvw, 0.37)
    m = interior(d)
    tol = dict(fp64=TOL, mixed=1e-5, fp32=max(1e-5, 2 * ktot**2 * 2.0**-24))[precision]
    for name in ("ut", "vt", "wt"):
        err = normwise(out[name], ref[name], m)
        assert err < tol, f"{name}: {err:.3e}"
    if precision != "mixed":
        err = normwise(out["p"][d.kstart - 1:d.kend], ref["p"][d.kstart - 1:d.kend])
        assert err < tol, f"p: {err:.3e}"
