"""The work that programs have this library do, as cases that can be timed and
checked: what each is in hand with before the call (prepare), one pass through
the public entry points (run), and the same numbers in 64 bits from plain torch
(exact).

The kinds of work:

  step      one RK3 time step of a large-eddy simulation of the dry boundary
            layer, three calls of mhh_substep_exec with a fixed time step
            (halos, ghost levels, viscosity, tendencies, projection, update)
  tendency  the first half of a substep: halos, ghost levels and
            mhh_tendency_2i5_smag2_visc, with or without the surface model
  pressure  mhh_pres_2_exec, the projection on its own
  channel   one RK3 step of a channel flow: 2nd-order advection and diffusion,
            the fixed-flux force, the projection with the RK3 update
  operators one RK3 step by the single operators, as a program does that has
            more than one scalar (the second is flux-limited)
  ensemble  one adaptive time step of several models with a surface layer,
            batched (microhh_amd.model.Ensemble)

Fields are torch tensors that the library borrows; it works on torch's default
stream.  torch is imported first, so that both use one HIP runtime.
"""
import ctypes as C
import math

import numpy as np
import torch

from microhh_amd import abi, model

PRECISIONS = {"fp64": abi.MHH_FP64, "fp32": abi.MHH_FP32, "mixed": abi.MHH_MIXED}
THREF = 300.0
GRAV = 9.81
CS, TPR, VISC = 0.23, 1.0 / 3.0, 1.0e-5
CHANNEL_NU = 3.57e-4          # Re_tau of about 180 for unit half height and bulk velocity
Z0M = 0.1
IGC = 3


def listed():
    return [
        # the smallest grid in use (an ensemble's smallest member, a test): launches and latency
        dict(name="step 32x32x32 fp32", kind="step", itot=32, jtot=32, ktot=32, precision="fp32", zgrid="uniform"),
        # a coarse production grid whose sizes are no powers of two, one of them odd
        dict(name="step 90x75x60 fp64", kind="step", itot=90, jtot=75, ktot=60, precision="fp64", zgrid="uniform"),
        # an ordinary LES in the mixed mode, two different lengths
        dict(name="step 256x192x96 mixed", kind="step", itot=256, jtot=192, ktot=96, precision="mixed",
             zgrid="uniform"),
        # the benchmark of this repository
        dict(name="step 512x512x256 fp64", kind="step", itot=512, jtot=512, ktot=256, precision="fp64",
             zgrid="uniform"),
        # the large stretched grid of the benchmark in the mixed mode, with half its levels
        dict(name="step 1024x1024x192 mixed", kind="step", itot=1024, jtot=1024, ktot=192, precision="mixed",
             zgrid="stretched"),
        # the tendencies alone, for a program with its own time integration
        dict(name="tendency 384x320x160 fp64", kind="tendency", itot=384, jtot=320, ktot=160, precision="fp64",
             zgrid="uniform", surface=False),
        # the same with the surface layer's gradients and fluxes, a ragged grid
        dict(name="tendency 150x100x75 fp32", kind="tendency", itot=150, jtot=100, ktot=75, precision="fp32",
             zgrid="stretched", surface=True),
        # the projection of a program with other operators, ragged lengths
        dict(name="pressure 360x250x100 fp32", kind="pressure", itot=360, jtot=250, ktot=100, precision="fp32",
             zgrid="uniform"),
        # the turbulent channel of the benchmark
        dict(name="channel 768x384x256 fp64", kind="channel", itot=768, jtot=384, ktot=256, precision="fp64",
             zgrid="tanh"),
        # a small channel, for statistics over long times
        dict(name="channel 192x96x64 mixed", kind="channel", itot=192, jtot=96, ktot=64, precision="mixed",
             zgrid="tanh"),
        # a moist-style set-up: two scalars, the second advected with the flux limiter
        dict(name="operators 240x180x120 fp64", kind="operators", itot=240, jtot=180, ktot=120, precision="fp64",
             zgrid="uniform"),
        # an ensemble of uneven members, three of each of the benchmark's four sizes
        dict(name="ensemble 12 fp32", kind="ensemble", each=3, base=32, precision="fp32"),
    ]


def member_sizes(case):
    n = case["base"]
    return [(n, n, n), (2 * n, 2 * n, 3 * n // 2), (3 * n, 3 * n, 2 * n), (4 * n, 4 * n, 3 * n)] * case["each"]


def smooth(n, primes):
    for p in primes:
        while n % p == 0:
            n //= p
    return n == 1


def draw_length(rng, low, high):
    """A transform length: the radices go up to 13; most programs take even
    lengths of 2, 3 and 5, some take what their domain gives."""
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    ragged = rng.random() < 0.3
    while not (smooth(n, (2, 3, 5, 7, 11, 13)) if ragged else n % 2 == 0 and smooth(n, (2, 3, 5))):
        n += 1
    return n


def draw(rng):
    kind = rng.choice(["step", "step", "step", "tendency", "pressure", "channel", "operators", "ensemble"])
    precision = rng.choice(["fp64", "fp32", "mixed"])
    if kind == "ensemble":
        return dict(kind=kind, each=rng.randint(1, 4), base=draw_length(rng, 16, 36),
                    precision=rng.choice(["fp64", "fp32"]))
    while True:
        itot = draw_length(rng, 16, 1024)
        jtot = draw_length(rng, max(16, itot // 4), min(1024, 2 * itot))
        ktot = int(round(math.exp(rng.uniform(math.log(12), math.log(320)))))
        if itot * jtot * ktot <= 32e6:
            break
    case = dict(kind=kind, itot=itot, jtot=jtot, ktot=ktot, precision=precision)
    case["zgrid"] = "tanh" if kind == "channel" else rng.choice(["uniform", "stretched"])
    if kind == "tendency":
        case["surface"] = rng.random() < 0.5
    return case


# ---------------------------------------------------------------- the set-up

def levels(case):
    """The grid's heights and 1-D profiles with kgc ghost levels on each side,
    as Grid::calculate sets them."""
    K, kgc = case["ktot"], 2 if case["kind"] == "operators" else 1
    if case["zgrid"] == "tanh":
        zsize = 2.0
        zc = model.tanh_levels(K, zsize, 2.75)
    elif case["zgrid"] == "stretched":
        zc, zsize = model.stretched_levels(K, 5.0, K // 2, 1.02)
    else:
        zsize = 12.5 * K
        zc = 12.5 * (np.arange(K) + 0.5)
    n = K + 2 * kgc
    ks, ke = kgc, kgc + K
    z, zh, dz, dzh = np.zeros(n), np.zeros(n), np.zeros(n), np.zeros(n)
    z[ks:ke] = zc
    for g in range(1, kgc + 1):
        z[ks - g] = -z[ks + g - 1]
        z[ke + g - 1] = 2 * zsize - z[ke - g]
    zh[ks + 1:ke] = 0.5 * (z[ks:ke - 1] + z[ks + 1:ke])
    zh[ks], zh[ke] = 0.0, zsize
    for g in range(1, kgc + 1):
        zh[ks - g] = -zh[ks + g]
        if ke + g < n:
            zh[ke + g] = 2 * zsize - zh[ke - g]
    dzh[1:] = z[1:] - z[:-1]
    dzh[ks - 1] = dzh[ks + 1]
    dz[:-1] = zh[1:] - zh[:-1]
    dz[ks - 1], dz[ke] = dz[ks], dz[ke - 1]
    dz[-1] = dz[-1] if dz[-1] > 0 else dz[ke - 1]
    dz[0] = dz[0] if dz[0] > 0 else dz[ks]
    dzh[0] = dzh[0] if dzh[0] > 0 else dzh[ks + 1]
    return dict(kgc=kgc, z=z, zh=zh, dz=dz, dzh=dzh, dzi=1.0 / dz, dzhi=1.0 / dzh, zsize=zsize)


def spacing(case):
    if case["kind"] == "channel":
        return 4.0 * math.pi / case["itot"], 2.0 * math.pi / case["jtot"]
    return 50.0, 40.0


def time_step(case, lev):
    if case["kind"] == "channel":
        return 0.25 * min(spacing(case)) / 3.0
    return 0.03 * float(lev["dz"].min())


def torch_type(case):
    return torch.float64 if case["precision"] == "fp64" else torch.float32


def theta_offset(case):
    return THREF if case["precision"] == "mixed" else 0.0


def inputs(case, seed):
    """Interior fields in 64 bits, of values that the field type holds: a mean
    wind with divergence-free eddies of several sizes and noise, and a stable
    layer above a mixed one."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    K, J, I = case["ktot"], case["jtot"], case["itot"]
    lev = levels(case)
    kgc, zsize = lev["kgc"], lev["zsize"]
    dx, dy = spacing(case)
    z = torch.tensor(lev["z"][kgc:kgc + K], device="cuda").view(K, 1, 1)
    zh = torch.tensor(lev["zh"][kgc:kgc + K + 1], device="cuda").view(K + 1, 1, 1)
    x = torch.arange(I, device="cuda", dtype=torch.float64).view(1, 1, I) * (2 * math.pi / I)
    y = torch.arange(J, device="cuda", dtype=torch.float64).view(1, J, 1) * (2 * math.pi / J)
    ft = torch_type(case)

    def eddies(amp, at, noise):
        a = torch.rand((at.shape[0], J, I), generator=gen, device="cuda", dtype=torch.float32).to(torch.float64)
        a = (a - 0.5) * noise
        for n in (1, 2, 5):
            ph = torch.rand(2, generator=gen, device="cuda", dtype=torch.float32).to(torch.float64) * (2 * math.pi)
            a += (amp / n) * torch.sin(n * x + ph[0]) * torch.sin(n * y + ph[1]) * torch.sin((n * math.pi / zsize) * at)
        return a

    def held(a):
        return a.to(ft).to(torch.float64)

    f = {}
    size = 0.05 if case["kind"] == "channel" else 0.4
    # a potential at the corners (horizontal eddies) and one above the west
    # faces, zero at the walls (overturning ones)
    horizontal = eddies(size * min(I * dx, J * dy) / (2 * math.pi), z, 0.3 * size * min(dx, dy))
    overturning = eddies(size * min(I * dx / (2 * math.pi), zsize / math.pi), zh, 0.3 * size * float(lev["dz"].min()))
    overturning[0], overturning[-1] = 0.0, 0.0
    dz = torch.tensor(lev["dz"][kgc:kgc + K], device="cuda").view(K, 1, 1)
    u = (torch.roll(horizontal, -1, 1) - horizontal) / dy + (overturning[1:] - overturning[:-1]) / dz
    v = (horizontal - torch.roll(horizontal, -1, 2)) / dx
    f["w"] = held(((overturning - torch.roll(overturning, -1, 2)) / dx)[:-1])
    if case["kind"] == "channel":
        f["u"], f["v"] = held(u + 1.5 * (1 - (z - 1) ** 2)), held(v)
    else:
        f["u"], f["v"] = held(u + 4.0), held(v - 2.0)
        th = THREF + 0.006 * torch.clamp(z - 0.4 * zsize, min=0.0) + eddies(0.1, z, 0.1)
        f["s0"] = held(th - theta_offset(case))
        if case["kind"] == "operators":
            f["s1"] = held(torch.clamp(eddies(1e-3, z, 1e-3) + 5e-3 * torch.exp(-z / 400.0), min=0.0))
    if case["kind"] in ("tendency", "pressure"):
        for n in ("u", "v", "w", "s0"):
            f["t" + n] = held(eddies(2e-3, z, 1e-3))
        f["tw"][0] = 0.0
    if case.get("surface"):
        one = torch.rand((6, J, I), generator=gen, device="cuda", dtype=torch.float32).to(torch.float64)
        f["dudz"], f["dvdz"] = held(0.3 + 0.1 * one[0]), held(-0.15 + 0.1 * one[1])
        f["dbdz"] = held(-0.01 * one[2])
        f["u_fluxbot"], f["v_fluxbot"] = held(-0.1 * one[3]), held(0.05 * one[4])
        f["s_fluxbot"] = held(0.1 + 0.02 * one[5])
        f["z0m"] = held(torch.full((J, I), Z0M, device="cuda", dtype=torch.float64))
    return f


FIELDS = ("u", "v", "w", "ut", "vt", "wt", "p", "evisc", "tmp1", "tmp2")
PLANES = ("u_bot", "u_top", "u_gradbot", "u_gradtop", "u_fluxbot", "u_fluxtop",
          "v_bot", "v_top", "v_gradbot", "v_gradtop", "v_fluxbot", "v_fluxtop", "dudz", "dvdz", "dbdz", "z0m")
SPLANES = ("s_bot", "s_top", "s_gradbot", "s_gradtop", "s_fluxbot", "s_fluxtop")
SBOT, SGRADTOP = (301.0, 6.0e-3), (0.006, 0.0)


class Context:
    """A context of the operator interface and the tensors bound to it."""

    def __init__(self, case, seed):
        self.case, self.lib = case, abi.lib()
        lev = self.lev = levels(case)
        self.kgc = kgc = lev["kgc"]
        K, J, I = case["ktot"], case["jtot"], case["itot"]
        self.ns = {"channel": 0, "operators": 2}.get(case["kind"], 1)
        dx, dy = spacing(case)
        one = np.ones(K + 2 * kgc)
        self.host = dict(lev, rhoref=one, rhorefh=one, thref=THREF * one)
        ptr = {n: a.ctypes.data_as(abi.DP) for n, a in self.host.items() if isinstance(a, np.ndarray)}
        grid = abi.GridDesc(I, J, K, IGC, IGC, kgc, dx, dy, lev["zsize"],
                            *[ptr[n] for n in ("z", "zh", "dz", "dzh", "dzi", "dzhi", "rhoref", "rhorefh")])
        self.h = C.c_void_p()
        abi.check(self.lib.mhh_ctx_create(C.byref(grid), PRECISIONS[case["precision"]], None, C.byref(self.h)),
                  "mhh_ctx_create")
        if self.ns:
            abi.check(self.lib.mhh_set_scalar_offset(self.h, 0, theta_offset(case)), "mhh_set_scalar_offset")
            abi.check(self.lib.mhh_set_base_state(self.h, ptr["thref"], ptr["thref"]), "mhh_set_base_state")
        shape3, shape2 = (K + 2 * kgc, J + 2 * IGC, I + 2 * IGC), (J + 2 * IGC, I + 2 * IGC)
        ft = torch_type(case)
        self.t = {n: torch.zeros(shape3, dtype=ft, device="cuda") for n in FIELDS}
        self.t.update({n: torch.zeros(shape2, dtype=ft, device="cuda") for n in PLANES})
        for q in range(self.ns):
            self.t.update({n + str(q): torch.zeros(shape3, dtype=ft, device="cuda") for n in ("s", "st")})
            self.t.update({n + str(q): torch.zeros(shape2, dtype=ft, device="cuda") for n in SPLANES})
            self.t["s_bot%d" % q].fill_(SBOT[q] - (theta_offset(case) if q == 0 else 0.0))
            self.t["s_gradtop%d" % q].fill_(SGRADTOP[q])
        fs = abi.FieldSet()
        for n in FIELDS + PLANES:
            setattr(fs, n, self.t[n].data_ptr())
        fs.nscalars = self.ns
        for q in range(self.ns):
            for n in ("s", "st") + SPLANES:
                getattr(fs, n)[q] = self.t[n + str(q)].data_ptr()
        abi.check(self.lib.mhh_fields_bind(self.h, C.byref(fs)), "mhh_fields_bind")
        for n, a in inputs(case, seed).items():
            if n == "s_fluxbot":
                n = "s_fluxbot0"
            elif n[0] == "t":
                n = "st0" if n == "ts0" else n[1] + "t"
            if a.dim() == 3:
                self.interior(n).copy_(a)
            else:   # a plane and its periodic images
                self.t[n].copy_(torch.nn.functional.pad(a[None, None], (IGC,) * 4, mode="circular")[0, 0])
        each = C.c_int * abi.MHH_MAX_SCALARS
        self.bc = abi.BcDesc(abi.BC["noslip"], abi.BC["noslip" if case["kind"] == "channel" else "freeslip"],
                             each(*[abi.BC["flux" if case.get("surface") else "dirichlet"]] * 8),
                             each(*[abi.BC["neumann"]] * 8))
        self.smag = abi.SmagParams(CS, TPR, VISC, (C.c_double * abi.MHH_MAX_SCALARS)(*[VISC] * 8), 1,
                                   1 if case.get("surface") else 0, 1)
        self.dt = time_step(case, lev)
        self.sub = [abi.SubstepDesc(self.smag, self.bc, 1, self.dt * part, s, self.dt,
                                    abi.MHH_RK3_SCALARS | abi.MHH_RK3_DEFER) for s, part in enumerate(SUBSTEPS)]
        if case["kind"] == "operators":
            self.call("mhh_advec_2i5_set_fluxlimit", (C.c_int * 2)(0, 1), 2)

    def interior(self, name):
        k = self.kgc
        return self.t[name][k:-k, IGC:-IGC, IGC:-IGC]

    def call(self, name, *args):
        abi.check(getattr(self.lib, name)(self.h, *args), name)

    def __del__(self):
        if getattr(self, "h", None):
            torch.cuda.synchronize()
            self.lib.mhh_ctx_destroy(self.h)


SUBSTEPS = (1.0 / 3.0, 5.0 / 12.0, 1.0 / 4.0)     # of the time step, RK3


class Members:
    """Models with a surface layer, each with its own noise and heat flux."""

    def __init__(self, case, seed):
        self.streams = model.Ensemble.streams(1)
        self.models, self.ensemble = [], None
        sizes = member_sizes(case)
        for m, (i, j, k) in enumerate(sizes):
            c = model.dry_cbl_surface_case(itot=i, jtot=j, ktot=k, xsize=100.0 * i, ysize=100.0 * j, zsize=50.0 * k,
                                           sbot=0.02 + 0.18 * m / len(sizes), precision=PRECISIONS[case["precision"]],
                                           dtmax=10.0, rndseed=seed % 1000003 + m)
            self.models.append(model.Model(c, stream=self.streams[0]))
        self.ensemble = model.Ensemble(self.models, mode="batched")

    def __del__(self):
        torch.cuda.synchronize()
        if self.ensemble:
            self.ensemble.close()
        for m in self.models:
            m.close()
        model.Ensemble.destroy_streams(self.streams)


class Borrowed:
    """A field of a model as torch sees it; the tensor keeps the models alive."""

    def __init__(self, members, m, name):
        self.members = members
        kind = "<f8" if m.case["precision"] == abi.MHH_FP64 else "<f4"
        self.__cuda_array_interface__ = dict(shape=m.shape, typestr=kind, data=(m.field_ptr(name), False), version=2)


class Ensemble:
    def __init__(self, case, seed):
        self.case, self.members = case, Members(case, seed)
        self.fields = [torch.as_tensor(Borrowed(self.members, m, n), device="cuda")[1:-1, IGC:-IGC, IGC:-IGC]
                       for m in self.members.models for n in ("u", "v", "w", "th")]


def prepare(case, seed):
    return Ensemble(case, seed) if case["kind"] == "ensemble" else Context(case, seed)


def run(s):
    kind = s.case["kind"]
    if kind == "ensemble":
        s.members.ensemble.steps(1)
        return s.fields
    if kind == "step":
        for d in s.sub:
            s.call("mhh_substep_exec", C.byref(d))
        return {n: s.interior(n) for n in ("u", "v", "w", "s0", "evisc")}
    if kind == "tendency":
        s.call("mhh_boundary_set_prognostic_cyclic_bcs")
        s.call("mhh_boundary_set_ghost_cells", C.byref(s.bc))
        s.call("mhh_tendency_2i5_smag2_visc", C.byref(s.smag), 1)
        return {n: s.interior(n) for n in ("ut", "vt", "wt", "st0", "evisc")}
    if kind == "pressure":
        s.call("mhh_boundary_set_prognostic_cyclic_bcs")
        s.call("mhh_pres_2_exec", s.dt)
        return {n: s.interior(n) for n in ("ut", "vt", "wt", "p")}
    for n, part in enumerate(SUBSTEPS):
        s.call("mhh_boundary_set_prognostic_cyclic_bcs")
        s.call("mhh_boundary_set_ghost_cells", C.byref(s.bc))
        if kind == "channel":
            s.call("mhh_tendency_2_2", CHANNEL_NU, None)
            s.call("mhh_force_fixed_flux", 1.0, 0.0, s.dt * part)
            s.call("mhh_pres_2_exec_rk3", s.dt * part, n, s.dt, abi.MHH_RK3_SCALARS)
        else:
            s.call("mhh_diff_smag2_exec_viscosity", C.byref(s.smag))
            s.call("mhh_thermo_dry_exec")
            s.call("mhh_advec_2i5_exec")
            s.call("mhh_diff_smag2_exec", C.byref(s.smag))
            s.call("mhh_pres_2_exec", s.dt * part)
            s.call("mhh_timeloop_rk3", n, s.dt)
    return {n: s.interior(n) for n in (("u", "v", "w") if kind == "channel" else ("u", "v", "w", "s0", "s1", "evisc"))}


def work(case):
    """Fields read and written once per operator call that needs them, and the
    operations of the stencils and transforms.  A substep: u, v, w, theta and
    their tendencies in and out, evisc and p out."""
    if case["kind"] == "ensemble":
        pts = sum(i * j * k for i, j, k in member_sizes(case))
        logs = 13.0
    else:
        pts = case["itot"] * case["jtot"] * case["ktot"]
        logs = math.log2(case["itot"]) + math.log2(case["jtot"])
    transform = 5.0 * logs + 20.0
    passes, flops = {"step": (3 * 18, 3 * (620 + transform)), "tendency": (13, 600), "pressure": (10, transform + 20),
                     "channel": (3 * 13, 3 * (140 + transform)), "operators": (3 * 22, 3 * (700 + transform)),
                     "ensemble": (3 * 18, 3 * (620 + transform))}[case["kind"]]
    return dict(bytes=pts * passes * (8 if case["precision"] == "fp64" else 4), flops=pts * flops)


def tolerance(case):
    """About four times what a change of the order of the sums, or of the
    transforms' radices, shows.  Whole steps amplify it through the projection
    (the pressure is large against its gradient) and, in fp32, through theta,
    whose perturbation is small against its value."""
    kind, p = case["kind"], case["precision"]
    if p == "fp64":
        # the ensemble's time step is cut to whole nanoseconds
        return dict(rel=1e-8 if kind == "ensemble" else 1e-11)
    return dict(rel={"step": (2e-4, 1e-4), "tendency": (2e-3, 1e-4), "pressure": (6e-3, 6e-3), "channel": (4e-4, 4e-4),
                     "operators": (4e-4, 1e-4), "ensemble": (3e-3, 3e-3)}[kind][p == "mixed"])


# ------------------------------------------------------- the same in 64 bits

def at(a, di=0, dj=0):
    """The periodic neighbour (di, dj) of every point."""
    return torch.roll(a, (-dj, -di), (1, 2)) if di or dj else a


def mid(a, b):
    return 0.5 * (a + b)


def face(vel, s, order):
    """Flux at the face below each value, advected by vel: s(m) is the value m
    cells up from the face's upper cell."""
    if order == 2:
        return vel * mid(s(-1), s(0))
    if order == 4:
        return vel * (7 * (s(-1) + s(0)) - (s(-2) + s(1))) / 12 - vel.abs() * (3 * (s(0) - s(-1)) - (s(1) - s(-2))) / 12
    return (vel * (37 * (s(-1) + s(0)) - 8 * (s(-2) + s(1)) + (s(-3) + s(2))) / 60
            - vel.abs() * (10 * (s(0) - s(-1)) - 5 * (s(1) - s(-2)) + (s(2) - s(-3))) / 60)


def vertical_faces(mass, s, n):
    """Fluxes at faces 0 .. n of n values, lower order next to the walls, none
    through them; mass[f] is the mass flux at face f."""
    out = torch.zeros_like(mass)
    for order, faces in ((2, (1, n - 1)), (4, (2, n - 2))):
        for f in faces:
            out[f] = face(mass[f], lambda m: s[f + m], order)
    out[3:n - 2] = face(mass[3:n - 2], lambda m: s[3 + m:n - 2 + m], 6)
    return out


def koren(vel, s):
    """Koren's limited flux at the face below each value."""
    def up(num, d):
        eps = torch.finfo(torch.float64).eps
        r2 = 2 * num / (torch.copysign(torch.ones_like(d), d) * d.abs().clamp(min=eps))
        return torch.minimum(torch.minimum(r2, (1 + r2) / 3), torch.full_like(r2, 2.0)).clamp(min=0.0)
    plus = s(-1) + (0.5 * up(s(0) - s(-1), s(-1) - s(-2)) * (s(-1) - s(-2)) if s(-2) is not None else 0.0)
    minus = s(0) + (0.5 * up(s(-1) - s(0), s(0) - s(1)) * (s(0) - s(1)) if s(1) is not None else 0.0)
    return torch.where(vel >= 0, vel * plus, vel * minus)


class Exact:
    """The equations in 64 bits on interior arrays [k, j, i] (w: half levels
    0 .. ktot, zero at both walls)."""

    def __init__(self, case, seed):
        self.case = case
        lev, f = levels(case), inputs(case, seed)
        K, k0 = case["ktot"], lev["kgc"]
        self.K = K

        def prof(a, first, n):
            return torch.tensor(np.ascontiguousarray(a[k0 + first:k0 + first + n]), device="cuda").view(n, 1, 1)
        self.dz, self.dzi, self.dzhi = prof(lev["dz"], 0, K), prof(lev["dzi"], 0, K), prof(lev["dzhi"], 0, K + 1)
        self.z = prof(lev["z"], 0, K)
        self.dxi, self.dyi = (1.0 / d for d in spacing(case))
        self.dx, self.dy = spacing(case)
        self.dt = time_step(case, lev)
        self.bits = torch_type(case)
        self.u, self.v = f["u"], f["v"]
        self.w = torch.cat([f["w"], torch.zeros_like(f["w"][:1])])
        # theta as stored, relative to an offset: in flux form its advection differs
        # from that of the whole value by the divergence of the stored velocities
        self.s = [f[n] for n in ("s0", "s1") if n in f]
        self.ut, self.vt = (f.get("t" + n, torch.zeros_like(f["u"])) for n in ("u", "v"))
        self.wt = torch.cat([f["tw"], torch.zeros_like(f["tw"][:1])]) if "tw" in f else torch.zeros_like(self.w)
        self.st = [f.get("ts0", torch.zeros_like(a)) for a in self.s]
        self.sfc = f if case.get("surface") else None

    def held(self, x):
        """A constant as the field type holds it."""
        return float(torch.tensor(x, dtype=self.bits))

    def ghosts(self):
        """u, v and the scalars with a ghost level below and above."""
        top = -1.0 if self.case["kind"] == "channel" else 1.0
        self.gu, self.gv = (torch.cat([-a[:1], a, top * a[-1:]]) for a in (self.u, self.v))
        off = theta_offset(self.case)
        self.gs = []
        for q, a in enumerate(self.s):
            bot = self.held(SBOT[q] - (off if q == 0 else 0.0))
            low = a[:1] if self.sfc is not None else 2 * bot - a[:1]
            self.gs.append(torch.cat([low, a, a[-1:] + self.held(SGRADTOP[q]) / self.dzhi[-1:]]))

    def viscosity(self):
        u, v, w = self.gu, self.gv, self.w
        dxi, dyi = self.dxi, self.dyi
        uc, vc = u[1:-1], v[1:-1]
        xy = ((uc - at(uc, 0, -1)) * dyi + (vc - at(vc, -1, 0)) * dxi) ** 2          # at the corner i-1/2, j-1/2
        xz = (u[1:] - u[:-1]) * self.dzhi + (w - at(w, -1, 0)) * dxi                 # at i-1/2, face k
        yz = (v[1:] - v[:-1]) * self.dzhi + (w - at(w, 0, -1)) * dyi
        xz, yz = xz ** 2, yz ** 2
        s2 = 2 * (((at(uc, 1) - uc) * dxi) ** 2 + ((at(vc, 0, 1) - vc) * dyi) ** 2 + ((w[1:] - w[:-1]) * self.dzi) ** 2
                  + 0.125 * (xy + at(xy, 1) + at(xy, 0, 1) + at(xy, 1, 1))
                  + 0.125 * (xz[:-1] + at(xz[:-1], 1) + xz[1:] + at(xz[1:], 1))
                  + 0.125 * (yz[:-1] + at(yz[:-1], 0, 1) + yz[1:] + at(yz[1:], 0, 1))) + 1e-9
        n2 = GRAV / THREF * 0.5 * self.dzi * (self.gs[0][2:] - self.gs[0][:-2])
        mlen2 = (CS * (self.dx * self.dy * self.dz) ** (1.0 / 3.0)) ** 2
        if self.sfc is not None:
            wx, wy = ((w[:2] - at(w[:2], -1, 0)) * dxi) ** 2, ((w[:2] - at(w[:2], 0, -1)) * dyi) ** 2
            s2[0] = 2 * (((at(uc[:1], 1) - uc[:1]) * dxi) ** 2 + ((at(vc[:1], 0, 1) - vc[:1]) * dyi) ** 2
                         + ((w[1:2] - w[:1]) * self.dzi[:1]) ** 2
                         + 0.125 * (xy[:1] + at(xy[:1], 1) + at(xy[:1], 0, 1) + at(xy[:1], 1, 1))
                         + 0.5 * (self.sfc["dudz"] ** 2 + self.sfc["dvdz"] ** 2)
                         + 0.125 * (wx + at(wx, 1) + wy + at(wy, 0, 1)).sum(0, keepdim=True))[0] + 1e-9
            n2[0] = self.sfc["dbdz"]
            mlen2 = 1.0 / (1.0 / mlen2 + 1.0 / (0.4 * (self.z + self.sfc["z0m"])) ** 2)
        self.evisc = mlen2 * torch.sqrt(torch.maximum(s2 - n2 / TPR, 1e-9 * s2))

    def advect(self, s, vx, vy, mass, dzi):
        fx, fy = face(vx, lambda m: at(s, m), 6), face(vy, lambda m: at(s, 0, m), 6)
        fz = vertical_faces(mass, s, s.shape[0])
        return -(at(fx, 1) - fx) * self.dxi - (at(fy, 0, 1) - fy) * self.dyi - (fz[1:] - fz[:-1]) * dzi

    def advect_limited(self, s, vx, vy, w):
        fx, fy = koren(vx, lambda m: at(s, m)), koren(vy, lambda m: at(s, 0, m))
        fz = torch.zeros_like(w)
        n = self.K
        fz[2:n - 1] = koren(w[2:n - 1], lambda m: s[2 + m:n - 1 + m])
        fz[1] = koren(w[1], lambda m: None if m == -2 else s[1 + m])
        fz[n - 1] = koren(w[n - 1], lambda m: None if m == 1 else s[n - 1 + m])
        return -(at(fx, 1) - fx) * self.dxi - (at(fy, 0, 1) - fy) * self.dyi - (fz[1:] - fz[:-1]) * self.dzi

    def les_tendencies(self):
        self.ghosts()
        self.viscosity()
        u, v, w, dxi, dyi = self.u, self.v, self.w, self.dxi, self.dyi
        # buoyancy on the half levels between the walls
        self.wt[1:-1] += GRAV / THREF * (mid(self.s[0][:-1], self.s[0][1:]) - (THREF - theta_offset(self.case)))
        self.ut += self.advect(u, mid(at(u, -1), u), mid(at(v, -1), v), mid(at(w, -1), w), self.dzi)
        self.vt += self.advect(v, mid(at(u, 0, -1), u), mid(at(v, 0, -1), v), mid(at(w, 0, -1), w), self.dzi)
        for q, s in enumerate(self.s):
            self.st[q] += self.advect(s, u, v, w, self.dzi) if q == 0 else self.advect_limited(s, u, v, w)
        # w on the half levels 0 .. K: the faces above and below them are the cell centres
        um, vm = (torch.cat([a[:1], mid(a[:-1], a[1:])]) for a in (u, v))
        wl = w[:-1]
        fx, fy = face(um, lambda m: at(wl, m), 6), face(vm, lambda m: at(wl, 0, m), 6)
        fz = torch.zeros_like(wl)                 # centre c, between w[c] and w[c+1]
        K = self.K
        mass = mid(w[:-1], w[1:])
        for order, cs in ((2, (0, K - 1)), (4, (1, K - 2))):
            for c in cs:
                fz[c] = face(mass[c], lambda m: w[c + 1 + m], order)
        fz[2:K - 2] = face(mass[2:K - 2], lambda m: w[3 + m:K - 1 + m], 6)
        adv = -(at(fx, 1) - fx) * dxi - (at(fy, 0, 1) - fy) * dyi
        self.wt[1:-1] += adv[1:] - (fz[1:] - fz[:-1]) * self.dzhi[1:-1]
        # diffusion
        ev = self.evisc
        ge = torch.cat([ev[:1], ev, ev[-1:]])
        gu, gv = self.gu, self.gv
        corner = 0.25 * (ev + at(ev, -1) + at(ev, 0, -1) + at(ev, -1, -1)) + VISC
        xy = corner * ((u - at(u, 0, -1)) * dyi + (v - at(v, -1)) * dxi)
        ex = 0.25 * (ge[1:] + ge[:-1] + at(ge[1:] + ge[:-1], -1)) + VISC          # i-1/2, face k
        ey = 0.25 * (ge[1:] + ge[:-1] + at(ge[1:] + ge[:-1], 0, -1)) + VISC
        xz = ex * ((gu[1:] - gu[:-1]) * self.dzhi + (w - at(w, -1)) * dxi)
        yz = ey * ((gv[1:] - gv[:-1]) * self.dzhi + (w - at(w, 0, -1)) * dyi)
        wxz, wyz = xz[1:-1], yz[1:-1]
        if self.sfc is not None:
            xz, yz = xz.clone(), yz.clone()
            xz[0], yz[0], xz[-1], yz[-1] = -self.sfc["u_fluxbot"], -self.sfc["v_fluxbot"], 0.0, 0.0
        uu = (ev + VISC) * (at(u, 1) - u) * dxi
        vv = (ev + VISC) * (at(v, 0, 1) - v) * dyi
        ww = (ev + VISC) * (w[1:] - w[:-1]) * self.dzi
        self.ut += 2 * (uu - at(uu, -1)) * dxi + (at(xy, 0, 1) - xy) * dyi + (xz[1:] - xz[:-1]) * self.dzi
        self.vt += 2 * (vv - at(vv, 0, -1)) * dyi + (at(xy, 1) - xy) * dxi + (yz[1:] - yz[:-1]) * self.dzi
        self.wt[1:-1] += (at(wxz, 1) - wxz) * dxi + (at(wyz, 0, 1) - wyz) * dyi \
            + 2 * (ww[1:] - ww[:-1]) * self.dzhi[1:-1]
        for q, s in enumerate(self.s):
            gs = self.gs[q]
            fx = (mid(ev, at(ev, -1)) / TPR + VISC) * (s - at(s, -1)) * dxi
            fy = (mid(ev, at(ev, 0, -1)) / TPR + VISC) * (s - at(s, 0, -1)) * dyi
            fz = (mid(ge[1:], ge[:-1]) / TPR + VISC) * (gs[1:] - gs[:-1]) * self.dzhi
            if self.sfc is not None:
                fz[0], fz[-1] = -self.sfc["s_fluxbot"], 0.0
            self.st[q] += (at(fx, 1) - fx) * dxi + (at(fy, 0, 1) - fy) * dyi + (fz[1:] - fz[:-1]) * self.dzi

    def channel_tendencies(self, dt):
        self.ghosts()
        u, v, w, dxi, dyi = self.u, self.v, self.w, self.dxi, self.dyi
        gu, gv = self.gu, self.gv

        def flux2(s, vx, vy):
            fx, fy = vx * mid(at(s, -1), s), vy * mid(at(s, 0, -1), s)
            return -(at(fx, 1) - fx) * dxi - (at(fy, 0, 1) - fy) * dyi

        def spread(s):
            return (at(s, 1) - 2 * s + at(s, -1)) * dxi ** 2 + (at(s, 0, 1) - 2 * s + at(s, 0, -1)) * dyi ** 2

        for a, g, t, d in ((u, gu, self.ut, (-1, 0)), (v, gv, self.vt, (0, -1))):
            fz = mid(at(w, *d), w) * mid(g[:-1], g[1:]) - CHANNEL_NU * (g[1:] - g[:-1]) * self.dzhi
            t += flux2(a, mid(at(u, *d), u), mid(at(v, *d), v)) + CHANNEL_NU * spread(a) - (fz[1:] - fz[:-1]) * self.dzi
        wi = w[1:-1]
        fz = mid(w[:-1], w[1:]) ** 2 - CHANNEL_NU * (w[1:] - w[:-1]) * self.dzi
        self.wt[1:-1] += flux2(wi, mid(u[:-1], u[1:]), mid(v[:-1], v[1:])) + CHANNEL_NU * spread(wi) \
            - (fz[1:] - fz[:-1]) * self.dzhi[1:-1]
        zsize = self.dz.sum()
        mean = [(a.mean((1, 2), keepdim=True) * self.dz).sum() / zsize for a in (u, self.ut)]
        self.ut += (1.0 - mean[0]) / dt - mean[1]

    def project(self, dt):
        hu, hv, hw = (t + a / dt for t, a in ((self.ut, self.u), (self.vt, self.v), (self.wt, self.w)))
        rhs = (at(hu, 1) - hu) * self.dxi + (at(hv, 0, 1) - hv) * self.dyi + (hw[1:] - hw[:-1]) * self.dzi
        K, J, I = rhs.shape
        q = torch.fft.rfft2(rhs) * self.dz ** 2
        kx = torch.arange(I // 2 + 1, device="cuda", dtype=torch.float64) * (2 * math.pi / I)
        ky = torch.arange(J, device="cuda", dtype=torch.float64) * (2 * math.pi / J)
        lam = -4 * ((torch.sin(0.5 * kx) * self.dxi) ** 2 + ((torch.sin(0.5 * ky) * self.dyi) ** 2)[:, None])
        dz, dzhi = self.dz.view(-1).tolist(), self.dzhi.view(-1).tolist()
        a, c = [dz[k] * dzhi[k] for k in range(K)], [dz[k] * dzhi[k + 1] for k in range(K)]
        gam = [None] * K
        piv = None
        for k in range(K):
            b = lam * dz[k] ** 2 - (a[k] + c[k])
            if k == 0:
                b = b + a[0]
            if k == K - 1:
                b = b + c[k]
                b[0, 0] -= 2 * c[k]
            if k:
                gam[k] = c[k - 1] / piv
                piv = b - a[k] * gam[k]
                q[k] = (q[k] - a[k] * q[k - 1]) / piv
            else:
                piv = b
                q[0] = q[0] / piv
        for k in range(K - 2, -1, -1):
            q[k] -= gam[k + 1] * q[k + 1]
        p = self.p = torch.fft.irfft2(q, s=(J, I))
        del q, gam
        self.ut -= (p - at(p, -1)) * self.dxi
        self.vt -= (p - at(p, 0, -1)) * self.dyi
        self.wt[1:-1] -= (p[1:] - p[:-1]) * self.dzhi[1:-1]

    def advance(self, n):
        cb, ca = (1 / 3, 15 / 16, 8 / 15)[n] * self.dt, (-5 / 9, -153 / 128, 0.0)[n]
        for a, t in [(self.u, self.ut), (self.v, self.vt), (self.w, self.wt)] + list(zip(self.s, self.st)):
            a += cb * t
            t *= ca


def exact(case, seed):
    """What run returns on a new state.  None for the ensemble: its surface
    layer is defined through a table in single precision, and its time step
    through whole nanoseconds."""
    kind = case["kind"]
    if kind == "ensemble":
        return None
    e = Exact(case, seed)
    if kind == "tendency":
        e.les_tendencies()
        return dict(ut=e.ut, vt=e.vt, wt=e.wt[:-1], st0=e.st[0], evisc=e.evisc)
    if kind == "pressure":
        e.project(e.dt)
        p = e.p - e.p.mean((1, 2), keepdim=True) if case["precision"] == "mixed" else e.p
        return dict(ut=e.ut, vt=e.vt, wt=e.wt[:-1], p=p)
    for n, part in enumerate(SUBSTEPS):
        if kind == "channel":
            e.channel_tendencies(e.dt * part)
        else:
            e.les_tendencies()
        e.project(e.dt * part)
        e.advance(n)
    out = dict(u=e.u, v=e.v, w=e.w[:-1])
    if kind != "channel":
        out.update({"s%d" % q: s for q, s in enumerate(e.s)}, evisc=e.evisc)
    return out
