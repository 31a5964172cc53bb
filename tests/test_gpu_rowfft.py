"""Transforms by lane groups at the lengths where their plan changes: one to
several passes, every radix and both kinds of butterflies, rows that do not fill a
group, odd numbers of rows (a pair with one row), the instance with 32 values
per lane (864, 1000, 1200, 1536), and a length without a plan (1050).  Few rows take 64
lanes each; NARROW holds grids with enough rows for 8, 16 and 32 lanes, several
rows to a wave and a last wave that is partly idle (tests/test_dispatch_cpu.py checks that
their plans are these).  FALLBACK: x and y transforms of lengths without a plan.

Against the oracle, normwise.  FP64: 1e-12 as for every pressure test.  FP32 and
mixed: 1e-5, the bound of the FP32 transforms in test_gpu_fft_sizes.py.  Both up to
512 points and in proportion to the length above: p is rounded by eps |p|, and against
the gradient of its largest wave, 2 pi |p| / (n dx), the difference of two
neighbours is off by a relative eps n / (2 pi) (FP32 2e-5 at 2048 points); the smallest
eigenvalue, a difference of 1 and cos(2 pi / n), loses digits with n as well, so the same
factor is used for p.  Plain FP32: its sweeps of up to K = 9 levels amplify roundings
by at most about K^2, and 81 times 6e-8 is half of 1e-5.  On long rows it carries a p that
is large against its gradient, the mean above all, through its transforms.  A pass of
radix R sums R products with rounded roots, (R + 2) 2^-24 of the largest value;
a p has gone through the passes of both lengths forward and inverse, and a tendency takes the
difference of two p: 4 sum (R + 2) 2^-24 max|p| / spacing, the bound where that is more
(the sum over the prime factors of both lengths, which is no less than over the radices).
"""
import pytest

from tests._golden import interior, normwise
from tests.test_gpu_fft_sizes import TOL, _gpu_pres, _oracle_pres

pytestmark = pytest.mark.gpu

SIZES = [(4, 6, 6), (13, 11, 6), (33, 16, 7), (75, 90, 9), (77, 26, 6), (96, 50, 6), (250, 36, 6), (360, 21, 6),
         (864, 8, 6), (12, 1000, 6), (960, 12, 6), (10, 1024, 6), (20, 686, 6), (6, 1050, 6), (1200, 8, 6), (6, 1536, 6),
         (32, 24, 160)]


def _longer(itot, jtot):
    return max(1.0, max(itot, jtot) / 512.0)


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
        assert err < TOL * _longer(itot, jtot), f"{name}: {err:.3e}"
    err = normwise(out["p"][d.kstart - 1:d.kend], ref["p"][d.kstart - 1:d.kend])
    assert err < TOL * _longer(itot, jtot), f"p: {err:.3e}"


# itot, jtot, ktot, lanes and butterflies of the x transform, the same of the y transform
NARROW = [(15, 637, 52, "8 radix8", "64 direct"), (14, 625, 53, "8 direct", "64 radix8"),
          (600, 15, 55, "64 radix8", "8 radix8"), (600, 13, 55, "64 radix8", "8 direct"),
          (12, 315, 57, "16 radix8", "64 direct"), (315, 14, 57, "64 direct", "16 direct"),
          (24, 175, 47, "32 radix8", "64 direct"), (175, 24, 47, "64 direct", "32 radix8")]
# the same with 9 levels, for plain FP32
NARROW32 = [(15, 3645, 9, "8 radix8", "none"), (14, 3645, 9, "8 direct", "none"), (12, 1875, 9, "16 radix8", "none"),
            (24, 945, 9, "32 radix8", "64 direct")]


def _passes(*lengths):
    total = 0
    for n in lengths:
        for q in (2, 3, 5, 7, 11, 13):
            while n % q == 0:
                n //= q
                total += q + 2
    return total


def _check(itot, jtot, ktot, precision):
    import numpy as np
    from microhh_amd import abi
    p, i = _case(itot, jtot, ktot)
    out, uvw = _gpu_pres(p, i, 0.37, generic=True,
                         precision=dict(fp64=abi.MHH_FP64, fp32=abi.MHH_FP32, mixed=abi.MHH_MIXED)[precision])
    d, ref = _oracle_pres(p, i, uvw, 0.37)
    m = interior(d)
    for name, spacing in (("ut", p["dx"]), ("vt", p["dy"]), ("wt", np.min(i["dz"]))):
        bound = (TOL if precision == "fp64" else 1e-5) * _longer(itot, jtot)
        if precision == "fp32":
            rounding = 4 * _passes(itot, jtot) * 2.0**-24 * np.abs(ref["p"][m]).max() / spacing
            bound = max(bound, rounding / np.abs(ref[name][m]).max())
        err = normwise(out[name], ref[name], m)
        assert err < bound, f"{name}: {err:.3e}, bound {bound:.3e}"


@pytest.mark.parametrize("itot,jtot,ktot,precision",
                         [(*s[:3], q) for s in NARROW for q in ("fp64", "mixed")] + [(*s[:3], "fp32") for s in NARROW32])
def test_several_rows_per_wave(itot, jtot, ktot, precision):
    _check(itot, jtot, ktot, precision)


# in x with an odd and an even length and an odd number of rows, and in y
FALLBACK = [(1050, 9, 6), (1485, 7, 6), (6, 1050, 6)]


@pytest.mark.parametrize("precision", ["fp64", "fp32", "mixed"])
@pytest.mark.parametrize("itot,jtot,ktot", FALLBACK)
def test_lengths_without_a_plan(itot, jtot, ktot, precision):
    _check(itot, jtot, ktot, precision)


ROWS32 = [(13, 11, 6), (75, 90, 9), (250, 36, 6), (64, 16, 7)]


@pytest.mark.parametrize("itot,jtot,ktot,precision",
                         [(*r, q) for q in ("mixed", "fp32") for r in ROWS32]
                         + [(864, 8, 6, "mixed"), (10, 960, 6, "mixed"), (2048, 6, 6, "mixed")])
def test_single_precision_rows(itot, jtot, ktot, precision):
    from microhh_amd import abi
    p, i = _case(itot, jtot, ktot)
    out, uvw = _gpu_pres(p, i, 0.37, generic=True, precision=abi.MHH_MIXED if precision == "mixed" else abi.MHH_FP32)
    d, ref = _oracle_pres(p, i, uvw, 0.37)
    m = interior(d)
    for name in ("ut", "vt", "wt"):
        err = normwise(out[name], ref[name], m)
        assert err < 1e-5 * _longer(itot, jtot), f"{name}: {err:.3e}"


@pytest.mark.parametrize("precision", ["fp64", "fp32", "mixed"])
def test_odd_last_row_is_transformed_alone(precision):
    """The x transforms pack two real rows into one complex row; the last row of
    an odd number has no partner and is packed with zero.  One row of four
    points: its cosine wave (points 0 and 2) and its sine wave (1 and 3) are the
    real and the imaginary part of one bin, and no sum of the transforms or of the
    sweep mixes them, so the small sine wave must come out the same with a large cosine
    wave beside it, to a few roundings of its own.  Packed with a copy of itself
    the row's two parts are added, and the sine wave is lost to the
    rounding of the cosine wave: 5e-6 of it in FP64, 6e-4 in FP32."""
    import numpy as np
    from microhh_amd import abi
    from tests._gpu import GpuCase
    K, igc, jgc, kgc, dx, dz = 6, 3, 1, 1, 50.0, 20.0
    n = K + 2 * kgc
    one = np.ones(n)
    grid = dict(z=(np.arange(n) - 0.5) * dz, zh=(np.arange(n) - 1.0) * dz, dz=dz * one, dzh=dz * one, dzi=one / dz,
                dzhi=one / dz, rhoref=one, rhorefh=one)
    large, eps = (3 * 2.0**36, 2.0**-53) if precision == "fp64" else (3 * 2.0**14, 2.0**-24)
    small = 5.0
    p = {}
    for big in (0.0, large):
        g = GpuCase(4, 1, K, igc, jgc, kgc, dx, dx, grid, nscalars=1,
                    precision=dict(fp64=abi.MHH_FP64, fp32=abi.MHH_FP32, mixed=abi.MHH_MIXED)[precision])
        try:
            ut = np.zeros(g.shape3)
            # differences along x: big, small, -big, -small
            ut[kgc + 2, jgc, igc:igc + 4] = (0.0, big, big + small, small)
            g.put("ut", ut)
            g.call("mhh_boundary_cyclic", g.ptr("ut"), 2)
            g.call("mhh_pres_2_exec", 1.0)
            p[big] = g.get("p")[kgc:-kgc, jgc, igc:igc + 4]
        finally:
            g.close()
    assert np.abs(p[large][:, 0]).min() > 1e3 * np.abs(p[0.0][:, 1]).max() > 0
    off = np.abs(p[large][:, 1::2] - p[0.0][:, 1::2]).max() / np.abs(p[0.0][:, 1::2]).max()
    assert off < 8 * eps, f"{off:.3e}"
