"""Pressure projection at transform lengths that have specialised kernels
(128, 256 and 512 points along x and y, with 7, 9 and 17 levels) against the
oracle, and the
specialised kernels against the general transforms (MHH_FFT_GENERIC=1) on the
same inputs.  FP64; tolerance 1e-12 normwise, as for every pressure test.
"""
import os

import numpy as np
import pytest

from oracle import pyoracle as po
from tests._golden import interior, normwise

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _c(a):
    return np.ascontiguousarray(a, dtype=np.float64).copy()


# Levels per length: the fused y/tridiagonal kernels take the levels in
# groups of R = n/64 (2, 4, 8), prefetching the next group while solving the
# current one; these counts cross at least two group boundaries and end on a
# partial group.
KTOT = {128: 7, 256: 9, 512: 17}


def _inputs(n, seed):
    from tests.golden.make_golden import make_inputs
    return make_inputs(dict(itot=n, jtot=n, ktot=KTOT[n], stretch=True, anelastic=True, dx=50.0, dy=40.0,
                            seed=seed))


def _gpu_pres(p, i, dt, generic, precision=None, split=False):
    """The projection on the GPU; generic: the general transform engine only;
    split: y transforms and tridiagonal sweep as three passes instead of the
    two fused ones (both switches are read when the context is created)."""
    from microhh_amd import abi
    from tests._gpu import GpuCase
    env = {"MHH_FFT_GENERIC": "1" if generic else "0", "MHH_YTRI_SPLIT": "1" if split else "0"}
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        g = GpuCase(p["itot"], p["jtot"], p["ktot"], p["igc"], p["jgc"], p["kgc"], p["dx"], p["dy"], i,
                    nscalars=1, precision=abi.MHH_FP64 if precision is None else precision)
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v
    try:
        for n in ("u", "v", "w", "ut", "vt", "wt"):
            g.put(n, i[n])
        for n in ("u", "v", "w"):
            g.call("mhh_boundary_cyclic", g.ptr(n), 2)
        u, v, w = g.get("u"), g.get("v"), g.get("w")
        g.call("mhh_pres_2_exec", dt)
        return {n: g.get(n) for n in ("ut", "vt", "wt", "p")}, (u, v, w)
    finally:
        g.close()


def _oracle_pres(p, i, uvw, dt):
    d = po.dims(p["itot"], p["jtot"], p["ktot"], p["igc"], p["jgc"], p["kgc"],
                p["dx"] * p["itot"], p["dy"] * p["jtot"], float(i["zh"][p["kgc"] + p["ktot"]]))
    L = po.lib()
    u, v, w = (_c(a) for a in uvw)
    ut, vt, wt = _c(i["ut"]), _c(i["vt"]), _c(i["wt"])
    pf, tmp1, tmp2 = np.zeros_like(ut), np.zeros_like(ut), np.zeros_like(ut)
    bmati, bmatj = np.zeros(d.itot), np.zeros(d.jtot)
    a, c = np.zeros(d.kmax), np.zeros(d.kmax)
    L.mo_pres_2_set_values(d, po.ptr(bmati), po.ptr(bmatj), po.ptr(a), po.ptr(c), po.ptr(_c(i["dz"])),
                           po.ptr(_c(i["dzhi"])), po.ptr(_c(i["rhorefh"])))
    L.mo_pres_2_input(d, po.ptr(pf), po.ptr(u), po.ptr(v), po.ptr(w), po.ptr(ut), po.ptr(vt), po.ptr(wt),
                      po.ptr(_c(i["dzi"])), po.ptr(_c(i["rhoref"])), po.ptr(_c(i["rhorefh"])), dt)
    L.mo_pres_2_solve(d, po.ptr(pf), po.ptr(tmp1), po.ptr(tmp2), po.ptr(_c(i["dz"])), po.ptr(_c(i["rhoref"])),
                      po.ptr(bmati), po.ptr(bmatj), po.ptr(a), po.ptr(c))
    L.mo_pres_2_output(d, po.ptr(ut), po.ptr(vt), po.ptr(wt), po.ptr(pf), po.ptr(_c(i["dzhi"])))
    return d, {"ut": ut, "vt": vt, "wt": wt, "p": pf}


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("n", [128, 256, 512])
def test_pres_specialised_lengths(n, split):
    p, i = _inputs(n, seed=31 + n)
    dt = 0.41
    out, uvw = _gpu_pres(p, i, dt, generic=False, split=split)
    d, ref = _oracle_pres(p, i, uvw, dt)
    m = interior(d)
    for name in ("ut", "vt", "wt"):
        err = normwise(out[name], ref[name], m)
        assert err < TOL, f"n={n} {name}: {err:.3e}"
    ks, ke = d.kstart, d.kend
    err = normwise(out["p"][ks - 1:ke], ref["p"][ks - 1:ke])
    assert err < TOL, f"n={n} p: {err:.3e}"


@pytest.mark.parametrize("n", [128, 512])
def test_specialised_matches_general_engine(n):
    p, i = _inputs(n, seed=7 + n)
    dt = 0.29
    fast, _ = _gpu_pres(p, i, dt, generic=False)
    gen, _ = _gpu_pres(p, i, dt, generic=True)
    for name in ("ut", "vt", "wt", "p"):
        err = normwise(fast[name], gen[name])
        assert err < 1e-13, f"n={n} {name}: {err:.3e}"


@pytest.mark.parametrize("n", [256, 512])
@pytest.mark.parametrize("prec", ["mixed", "fp32"])
def test_float_specialised_matches_general_engine(prec, n):
    """The mixed mode (FP32 fields and transforms, FP64 plane means and
    tridiagonal) and plain FP32 through both transform engines: the same
    projection to FP32 rounding."""
    from microhh_amd import abi
    precision = abi.MHH_MIXED if prec == "mixed" else abi.MHH_FP32
    p, i = _inputs(n, seed=99)
    dt = 0.33
    fast, _ = _gpu_pres(p, i, dt, generic=False, precision=precision)
    gen, _ = _gpu_pres(p, i, dt, generic=True, precision=precision)
    for name in ("ut", "vt", "wt"):
        err = normwise(fast[name], gen[name])
        assert err < 1e-5, f"{name}: {err:.3e}"


# The instances of the general transforms (MHH_FFT_GENERIC): lane groups with 16
# values per lane and radices 8, 4, 2, 3, 5 (96 = 4 8 3, 768 = 4 8 8 3), with 32
# values (1000 = 8 5 5 5: radix-5 passes of 200 butterflies, 4 per lane), with
# butterflies by definition (56 = 8 7; 1300 = 4 5 5 13 with a radix-13 pass and a
# radix-4 pass of 325 butterflies), and the ping-pong transform in two row
# buffers of the lengths without a plan (1050 = 2 3 5 5 7, 1078 = 2 7 7 11).
@pytest.mark.parametrize("itot,jtot", [(96, 768), (1000, 12), (56, 1300), (1050, 9), (8, 1078)],
                         ids=["values16", "values32", "direct", "pingpong-x", "pingpong-y"])
def test_pres_general_engine_instances(itot, jtot):
    from tests.golden.make_golden import make_inputs
    p, i = make_inputs(dict(itot=itot, jtot=jtot, ktot=6, stretch=True, anelastic=True, dx=50.0, dy=40.0,
                            seed=itot + jtot))
    dt = 0.37
    out, uvw = _gpu_pres(p, i, dt, generic=True)
    d, ref = _oracle_pres(p, i, uvw, dt)
    m = interior(d)
    for name in ("ut", "vt", "wt"):
        err = normwise(out[name], ref[name], m)
        assert err < TOL, f"{itot}x{jtot} {name}: {err:.3e}"
    ks, ke = d.kstart, d.kend
    err = normwise(out["p"][ks - 1:ke], ref["p"][ks - 1:ke])
    assert err < TOL, f"{itot}x{jtot} p: {err:.3e}"
