"""The plane means in chunks of rows, through the calls that use them: the
fixed-flux force (mhh_force_fixed_flux, Force::exec with swlspres = uflux) and
the buffer with swupdate (mhh_buffer_exec).

Sizes: chunks of several rows with a shorter last one and rows of more than
256 points (330 x 208), rows just over and just under what a wave reads at a time
(260, 63), fewer rows than a block has waves, and more levels than the
fold of the force has threads (300).

Force, against numpy in FP64 on the values that the field holds: the means are
FP64 sums in another order, so FP64 fields agree to 1e-13 of the terms
of the force and FP32 fields to the rounding of the sum ut + fbody, 2^-24 of either
(2^-23 here).  Buffer, against the oracle: 1e-12 normwise, all fields of a call.
"""
import ctypes as C
import time

import numpy as np
import pytest

from oracle import pyoracle as po
from tests._golden import normwise

pytestmark = pytest.mark.gpu

SIZES = [(330, 208, 60), (260, 5, 6), (63, 4, 9), (24, 9, 300)]


def _case(itot, jtot, ktot, nscalars, precision):
    from tests._gpu import GpuCase
    d = po.dims(itot, jtot, ktot, 3, 3, 1, 50.0 * itot, 50.0 * jtot, 20.0 * ktot)
    s = (np.arange(ktot) + 0.5) / ktot
    g = po.grid_arrays(d, 20.0 * ktot * s * (0.6 + 0.4 * s))
    g["rhoref"] = po.prof(d, 1.0)
    g["rhorefh"] = po.prof(d, 1.0)
    return d, g, GpuCase(itot, jtot, ktot, 3, 3, 1, 50.0, 50.0, g, nscalars=nscalars, precision=precision)


def _precision(name):
    from microhh_amd import abi
    return dict(fp64=abi.MHH_FP64, fp32=abi.MHH_FP32, mixed=abi.MHH_MIXED)[name]


@pytest.mark.parametrize("precision", ["fp64", "fp32", "mixed"])
@pytest.mark.parametrize("itot,jtot,ktot", SIZES)
def test_fixed_flux_force(itot, jtot, ktot, precision):
    d, g, gc = _case(itot, jtot, ktot, 1, _precision(precision))
    rng = np.random.default_rng(itot)
    uflux, utrans, dt = 1.5, 0.25, 0.7
    try:
        gc.put("u", 2.0 + rng.uniform(-1.0, 1.0, gc.shape3))
        gc.put("ut", rng.uniform(-1e-2, 1e-2, gc.shape3))
        u, ut = gc.get("u"), gc.get("ut")
        gc.call("mhh_force_fixed_flux", uflux, utrans, dt)
        got = gc.get("ut")
    finally:
        gc.close()
    inner = np.s_[d.kstart:d.kend, d.jstart:d.jend, d.istart:d.iend]
    dz, zsize = g["dz"][d.kstart:d.kend], g["zh"][d.kend]
    mean = [np.sum(a[inner].mean(axis=(1, 2)) * dz) / zsize for a in (u, ut)]
    fbody = (uflux - mean[0] - utrans) / dt - mean[1]
    ref = ut.copy()
    ref[inner] += fbody
    tol = 1e-13 * (uflux + abs(mean[0]) + utrans) / dt if precision == "fp64" else 2.0**-23 * (abs(fbody) + 1e-2)
    assert np.abs(got - ref).max() < tol
    assert np.array_equal(np.delete(got, np.s_[d.kstart:d.kend], 0), np.delete(ut, np.s_[d.kstart:d.kend], 0))


@pytest.mark.parametrize("itot,jtot,ktot", SIZES)
def test_buffer_means(itot, jtot, ktot):
    from microhh_amd import abi
    d, g, gc = _case(itot, jtot, ktot, 2, abi.MHH_FP64)
    L = po.lib()
    rng = np.random.default_rng(jtot)
    names = (("ut", "u"), ("vt", "v"), ("wt", "w"), ("st0", "s0"), ("st1", "s1"))
    try:
        f = {n: rng.uniform(-1.0, 1.0, gc.shape3) + q for q, pair in enumerate(names) for n in pair}
        for n, a in f.items():
            gc.put(n, a)
        zsize = float(g["zh"][d.kend])
        zstart, sigma, beta = 0.6 * zsize, 0.01, 2.0
        zero = np.zeros(d.kcells)
        sp = (abi.DP * 2)(*[zero.ctypes.data_as(abi.DP)] * 2)
        desc = abi.BufferDesc(zstart, sigma, beta, 1)
        gc.call("mhh_buffer_init", C.byref(desc), zero.ctypes.data_as(abi.DP), zero.ctypes.data_as(abi.DP), sp, 2)
        gc.call("mhh_buffer_exec")
        kb, kbh = C.c_int(), C.c_int()
        L.mo_buffer_levels(d, po.ptr(g["z"]), po.ptr(g["zh"]), zstart, C.byref(kb), C.byref(kbh))
        for tend, name in names:
            prof = po.prof(d)
            L.mo_mean_profile(d, po.ptr(prof), po.ptr(f[name]))
            ref = f[tend].copy()
            z, k0 = (g["zh"], kbh.value) if name == "w" else (g["z"], kb.value)
            L.mo_buffer(d, po.ptr(ref), po.ptr(f[name]), po.ptr(prof), po.ptr(z), zstart, zsize, beta, sigma, k0)
            err = normwise(gc.get(tend) - f[tend], ref - f[tend])
            assert err < 1e-12, f"{tend}: {err:.3e}"
    finally:
        gc.close()


def test_buffer_means_of_all_fields_in_one_pass():
    """On a small grid the time of the buffer is that of its launches: one with
    given profiles, two more with the means of all fields (2.4 to 3.5 times as
    long; with a pass and a fold per field it took 7.5 times as long)."""
    from microhh_amd import abi
    best = {}
    for swupdate in (0, 1):
        d, g, gc = _case(16, 16, 16, 1, abi.MHH_FP64)
        try:
            zero = np.zeros(d.kcells)
            p = zero.ctypes.data_as(abi.DP)
            desc = abi.BufferDesc(0.75 * float(g["zh"][d.kend]), 0.01, 2.0, swupdate)
            gc.call("mhh_buffer_init", C.byref(desc), p, p, (abi.DP * 1)(p), 1)
            times = []
            for _ in range(12):
                gc.call("mhh_sync")
                start = time.perf_counter()
                for _ in range(200):
                    gc.call("mhh_buffer_exec")
                gc.call("mhh_sync")
                times.append(time.perf_counter() - start)
            best[swupdate] = min(times)
        finally:
            gc.close()
    assert best[1] < 4.5 * best[0], best
