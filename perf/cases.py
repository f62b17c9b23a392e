"""What a user has this framework do, as cases that can be timed and checked.

Every case goes through the public entry points (`cosmograph_amd.BSSN` and
`Batch`, or the C call beside them where the program keeps its own output
buffers).  The kinds:

  evolve   the main path: an output interval of whole RK4 steps, then the
           fields are read back
  method   the drop-in form: stepInit, RKEvolve and K{n}Finalize one by one
  batch    an ensemble of independent boxes advanced together
  output   the diagnostics of an output step: constraint statistics, the
           curvature arrays, a strip, conformal statistics, power spectra
  svt      the SVT / Bardeen potentials of an output step
  ics      constraint-solved initial data from a half-spectrum of modes

Sizes are those of the repository's own runs (32^3 smoke runs, the 128^3 FP64
run, the 256^3 split-precision run, the 48^3..128^3 ensemble, the dust box) and
generic ragged ones.  `exact` restates each path in plain torch, FP64, with
periodic rolls.
"""
import ctypes
import math

import numpy as np
import torch

import cosmograph_amd as cg

PI = math.pi
RHO_BAR = 3.0 / (8.0 * PI)  # units H_I = 1
K_BAR = -math.sqrt(24.0 * PI * RHO_BAR)
LAMBDA = 0.7 * RHO_BAR      # the dust box's Lambda energy density

MET = ["DIFFgamma11", "DIFFgamma12", "DIFFgamma13", "DIFFgamma22", "DIFFgamma23", "DIFFgamma33"]
AIJ = ["A11", "A12", "A13", "A22", "A23", "A33"]
GAM = ["Gamma1", "Gamma2", "Gamma3"]
FIELDS = MET + ["DIFFphi"] + AIJ + ["DIFFK"] + GAM
BETA = ["beta1", "beta2", "beta3"]
AUXB = ["auxB1", "auxB2", "auxB3"]
DUST = ["dust_D", "dust_S1", "dust_S2", "dust_S3"]
SYM = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]


def _sy(a, b):
    return SYM.index((min(a, b), max(a, b)))


# ------------------------------------------------------------------ cases --
def listed():
    c = dict
    return [
        # the smallest runs: convergence tests and smoke runs, where launches and latency are all there is
        c(name="evolve_32_fp64", kind="evolve", nx=32, ny=32, nz=32, order=4, precision="fp64", matter="static",
          lapse="Static", shift="none", ko=0.0, steps=16),
        # the FP64 drop-in at its quoted size and order
        c(name="evolve_128_fp64", kind="evolve", nx=128, ny=128, nz=128, order=4, precision="fp64", matter="static",
          lapse="Static", shift="none", ko=0.0, steps=24),
        # the headline box: 256^3, 6th order, every perturbation field in four bytes
        c(name="evolve_256_fix", kind="evolve", nx=256, ny=256, nz=256, order=6, precision="fp32_fix",
          matter="static", lapse="Static", shift="none", ko=0.0, steps=40),
        # a ragged box (no extent a multiple of a tile, k not of four) in split precision
        c(name="evolve_ragged_split", kind="evolve", nx=101, ny=90, nz=118, order=6, precision="fp32_split",
          matter="static", lapse="Static", shift="none", ko=0.0, steps=24),
        # vacuum waves with an evolved lapse and Kreiss-Oliger dissipation: the reference's default order 8
        c(name="evolve_waves_o8", kind="evolve", nx=96, ny=96, nz=96, order=8, precision="fp64", matter="none",
          lapse="Harmonic", shift="none", ko=0.1, steps=12),
        # the dust fluid with Lambda, perturbations of the FRW fluids: the large production box's physics
        c(name="evolve_192_dust", kind="evolve", nx=192, ny=192, nz=192, order=6, precision="fp32_fix",
          matter="dust", lapse="Static", shift="none", ko=0.0, steps=24),
        # the shift build: 1+log lapse and Gamma driver, advection along both upwind directions
        c(name="evolve_112_shift", kind="evolve", nx=112, ny=112, nz=112, order=4, precision="fp64", matter="static",
          lapse="OnePlusLog", shift="GammaDriver", ko=0.0, steps=6),
        # a reference program ported call by call
        c(name="method_96_fp64", kind="method", nx=96, ny=96, nz=96, order=6, precision="fp64", matter="static",
          lapse="Static", shift="none", ko=0.0, steps=6),
        # an ensemble of small boxes of unequal sizes
        c(name="batch_16", kind="batch", small=48, many=10, middle=64, some=4, large=96, few=2, order=4,
          precision="fp32_split", steps=12),
        # the diagnostics of an output step of an FP64 run
        c(name="output_192_fp64", kind="output", nx=192, ny=192, nz=192, order=6, precision="fp64"),
        # the SVT potentials of an output step
        c(name="svt_128", kind="svt", nx=128, ny=128, nz=128, order=4, precision="fp64"),
        # starting a realisation
        c(name="ics_192", kind="ics", n=192, precision="fp64"),
    ]


def _size(rng, lo, hi, mult=1):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, n // mult * mult)


def draw(rng):
    kind = rng.choice(["evolve"] * 6 + ["method", "batch", "output", "svt", "ics"])
    if kind == "ics":
        return dict(kind=kind, n=_size(rng, 24, 200, 2), precision=rng.choice(["fp64", "fp32_split", "fp32_fix"]))
    if kind == "batch":
        return dict(kind=kind, small=_size(rng, 20, 56), many=rng.randint(2, 10), middle=_size(rng, 40, 72),
                    some=rng.randint(1, 4), large=_size(rng, 64, 96), few=rng.randint(1, 2), order=4,
                    precision=rng.choice(["fp64", "fp32_split"]), steps=rng.randint(2, 12))
    top = {"evolve": 180, "method": 96, "output": 176, "svt": 128}[kind]
    even = kind in ("output", "svt")
    n = _size(rng, 24, top)
    nx, ny = (max(20, int(n * rng.uniform(0.75, 1.0))) for _ in range(2))
    nz = max(24, int(n * rng.uniform(0.75, 1.0)))
    nz = nz // 2 * 2 if even else nz
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz, order=rng.choice([2, 4, 6, 8]), precision="fp64")
    if even:
        return case
    case.update(matter="static", lapse="Static", shift="none", ko=0.0, steps=rng.randint(2, 8))
    if kind == "method":
        return case
    what = rng.choice(["static", "static", "static", "waves", "dust", "shift"])
    if what == "static":
        case["precision"] = rng.choice(["fp64", "fp32_split", "fp32_all", "fp32_fix"])
        if case["precision"] in ("fp32_all", "fp32_fix"):
            case["order"] = rng.choice([4, 6])
    elif what == "waves":
        case.update(matter="none", lapse="Harmonic", ko=rng.choice([0.0, 0.1]),
                    precision=rng.choice(["fp64", "fp32_split"]))
    elif what == "dust":
        case.update(matter="dust", order=rng.choice([4, 6]), precision=rng.choice(["fp64", "fp32_split", "fp32_fix"]))
    else:
        case.update(lapse="OnePlusLog", shift="GammaDriver", order=rng.choice([4, 6]),
                    nx=min(nx, 112), ny=min(ny, 112), nz=min(nz, 112), steps=rng.randint(2, 6))
    return case


# ----------------------------------------------------------- initial data --
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rand(seed, *shape):
    return torch.randn(*shape, generator=_gen(seed), device="cuda", dtype=torch.float64)


def _lattice(shape):
    k = [torch.fft.fftfreq(n, d=1.0 / n, device="cuda", dtype=torch.float64) for n in shape[:2]]
    k.append(torch.fft.rfftfreq(shape[2], d=1.0 / shape[2], device="cuda", dtype=torch.float64))
    return torch.meshgrid(*k, indexing="ij")


def _modes(shape, seed, index=-3.0):
    """Half-spectrum of a Gaussian field, P(k) ~ k^index on 1 <= |k| <= N/4."""
    kx, ky, kz = _lattice(shape)
    k = torch.sqrt(kx * kx + ky * ky + kz * kz)
    shell = (k >= 1.0) & (k <= min(shape) / 4.0)
    amp = torch.where(shell, torch.where(shell, k, torch.ones_like(k)) ** (index / 2.0), torch.zeros_like(k))
    g = _rand(seed, 2, *k.shape)
    return amp * torch.complex(g[0], g[1])


def _solve(modes, shape, rms, dx):
    """Conformal factor and density of constraint-solved dust: lap(u) = -2 pi u^5 (drho - c), u = e^phi."""
    delta = torch.fft.irfftn(modes, s=shape)
    delta = delta - delta.mean()
    drho = RHO_BAR * delta * (rms / torch.sqrt((delta * delta).mean()))
    kx, ky, kz = _lattice(shape)
    w = [(2.0 * PI / (n * dx)) ** 2 for n in shape]
    k2 = w[0] * kx * kx + w[1] * ky * ky + w[2] * kz * kz
    inv = torch.where(k2 > 0, -1.0 / torch.where(k2 > 0, k2, torch.ones_like(k2)), torch.zeros_like(k2))
    u, c = torch.ones_like(drho), 0.0
    for _ in range(200):
        u5 = u ** 5
        c = float((u5 * drho).mean() / u5.mean())
        un = 1.0 + torch.fft.irfftn(torch.fft.rfftn(-2.0 * PI * u5 * (drho - c)) * inv, s=shape)
        d = float((un - u).abs().max())
        u = un
        if d < 1e-15:
            break
    phi = torch.log(u)
    return phi, torch.exp(6.0 * phi) * (RHO_BAR + drho - c), c


def _smooth(shape, seed, amp):
    """A few long periodic modes with random phases."""
    g = np.random.default_rng(seed)
    x = [torch.arange(n, device="cuda", dtype=torch.float64) / n for n in shape]
    out = torch.zeros(shape, device="cuda", dtype=torch.float64)
    for _ in range(4):
        k = g.integers(-2, 3, size=3)
        arg = 2 * PI * (k[0] * x[0][:, None, None] + k[1] * x[1][None, :, None] + k[2] * x[2][None, None, :])
        out += float(g.standard_normal()) * torch.cos(arg + float(g.uniform(0, 2 * PI)))
    return amp * out


def _shape(case):
    return (case["nx"], case["ny"], case["nz"])


def _start(case, seed):
    """Initial fields (name -> tensor) and FRW background of an evolved case."""
    shape, dx = _shape(case), 1.0 / case["nx"]
    if case["matter"] == "none":
        # two transverse traceless standing waves along each axis, and a slightly perturbed lapse
        f = {}
        g = np.random.default_rng(seed)
        for ax, (p, q, r) in enumerate([(3, 5, 4), (0, 5, 2), (0, 3, 1)]):
            n = shape[ax]
            x = (torch.arange(n, device="cuda", dtype=torch.float64) / n).reshape([n if d == ax else 1 for d in range(3)])
            for m in (1, 2):
                a, b, ph = g.uniform(1e-5, 2e-5), g.uniform(1e-5, 2e-5), g.uniform(0, 2 * PI)
                wave = torch.cos(2 * PI * m * x + ph).expand(shape)
                for name, s in ((MET[p], a), (MET[q], -a), (MET[r], b)):
                    f[name] = f.get(name, 0) + s * wave
        f["DIFFalpha"] = _smooth(shape, seed + 1, 1e-5)
        return f, dict(phi=0.0, K=0.0, fluids=[])
    # amplitudes of the repository's own runs; small enough in FP64 that a program may go on for 10^4 steps
    rms = 3e-2 if case["matter"] == "dust" else 1e-2 if _single(case) else 1e-3
    phi, D, _ = _solve(_modes(shape, seed), shape, rms, dx)
    f = {"DIFFphi": phi}
    if case["matter"] == "dust":
        f["dust_D"] = D
        for j in range(3):  # small peculiar velocities
            f[DUST[1 + j]] = D * _smooth(shape, seed + 2 + j, 1e-3)
        return f, dict(phi=0.0, K=-math.sqrt(24.0 * PI * (RHO_BAR + LAMBDA)), fluids=[(RHO_BAR, 0.0), (LAMBDA, -1.0)])
    if case["shift"] != "none":
        # the whole K in the field, no reference background; a smooth shift of either sign
        f.update(DIFFD=D, DIFFK=torch.full(shape, K_BAR, device="cuda", dtype=torch.float64))
        for m, b in enumerate(BETA):
            f[b] = _smooth(shape, seed + 2 + m, 1e-3)
        return f, dict(phi=0.0, K=0.0, fluids=[])
    f["DIFFD"] = D - RHO_BAR
    return f, dict(phi=0.0, K=K_BAR, fluids=[(RHO_BAR, 0.0)])


# ------------------------------------------------------------ the program --
def _params(case):
    lam = LAMBDA if case["matter"] == "dust" else 0.0
    return cg.GpuParams(n=_shape(case), order=case["order"], precision=case["precision"], matter=case["matter"],
                        lapse=case["lapse"], shift=case["shift"], ko_coeff=case["ko"], lambda_=lam,
                        gd_eta=1.0 if case["shift"] == "GammaDriver" else 0.0)


def _load(g, fields, frw):
    g.frw_set(frw["phi"], frw["K"])
    for rho, w in frw["fluids"]:
        g.frw_add_fluid(rho, w)
    for name, x in fields.items():
        g.upload(name + ("_a" if name == "DIFFD" else "_p"), x.cpu().numpy())


def _kept(case):
    """The fields an output interval reads back: all that evolve on grids up to 128^3, one of each kind beyond."""
    big = case["nx"] * case["ny"] * case["nz"] > 128 ** 3
    names = ["DIFFgamma11", "DIFFgamma12", "DIFFphi", "A11", "A12", "DIFFK", "Gamma1"] if big else list(FIELDS)
    if case["lapse"] != "Static":
        names.append("DIFFalpha")
    if case["shift"] != "none":
        names += BETA + AUXB
    if case["matter"] == "dust":
        names += ["dust_D", "dust_S1"] if big else DUST
    return names


class _Snapshot:
    """Output buffers a program keeps: pinned FP64 for the read, and FP32 copies where the run is stored in FP32."""

    def __init__(self, names, shape, single):
        self.n = int(np.prod(shape))
        self.b = {f: torch.empty(shape, dtype=torch.float64, pin_memory=True) for f in names}
        self.s = {f: torch.empty(shape, dtype=torch.float32, pin_memory=True) for f in names} if single else None

    def read(self, g, key=lambda f: f + "_p"):
        for f, b in self.b.items():
            rc = g.L.cg_field_download(g.h, key(f).encode(), ctypes.cast(b.data_ptr(), ctypes.POINTER(ctypes.c_double)),
                                       self.n)
            if rc:
                raise RuntimeError(g.L.cg_last_error(g.h).decode())
            if self.s:
                self.s[f].copy_(b)
        return dict(self.s or self.b)


def _single(case):
    return case["precision"] != "fp64"


def _members(case):
    return [case["small"]] * case["many"] + [case["middle"]] * case["some"] + [case["large"]] * case["few"]


def _member(case, n):
    return dict(nx=n, ny=n, nz=n, order=case["order"], precision=case["precision"], matter="static", lapse="Static",
                shift="none", ko=0.0, steps=case["steps"])


def _general(case, seed):
    """Every field a smooth random perturbation of flat space: all terms of the diagnostics are at work."""
    shape = _shape(case)
    f = {name: _smooth(shape, 100 * seed + i, 1e-3) for i, name in enumerate(FIELDS + ["DIFFalpha", "DIFFD"])}
    f["DIFFD"] = f["DIFFD"] + RHO_BAR
    f["DIFFK"] = f["DIFFK"] - 0.3  # an expanding box: the averages of K are numbers, not rounding
    return f


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("evolve", "method"):
        fields, frw = _start(case, seed)
        g = cg.BSSN(_params(case))
        if case["matter"] == "dust":
            g.set_dust_background(True)
        _load(g, fields, frw)
        return dict(case=case, g=g, out=_Snapshot(_kept(case), _shape(case), _single(case)))
    if kind == "batch":
        sizes = _members(case)
        b = cg.Batch([_params(_member(case, n)) for n in sizes])
        for r, n in enumerate(sizes):
            _load(b.members[r], *_start(_member(case, n), seed * 64 + r))
        outs = [_Snapshot(["DIFFphi", "DIFFK", "A12"], (n, n, n), _single(case)) for n in sizes]
        return dict(case=case, g=b, out=outs)
    if kind in ("output", "svt"):
        g = cg.BSSN(_params(dict(case, matter="static", lapse="Harmonic", shift="none", ko=0.0)))
        _load(g, _general(case, seed), dict(phi=0.0, K=0.0, fluids=[]))
        names = ["ricci", "AijAij"] if kind == "output" else ["Phi", "Psi", "B", "C1", "D11"]
        return dict(case=case, g=g, out=_Snapshot(names, _shape(case), False))
    n = case["n"]
    modes = _modes((n, n, n), seed).cpu().numpy()
    g = cg.BSSN(cg.GpuParams(n=n, order=6, precision=case["precision"], matter="static"))
    return dict(case=case, g=g, modes=modes, out=_Snapshot(["DIFFphi", "DIFFD"], (n, n, n), _single(case)))


def run(state):
    case, g, out = state["case"], state["g"], state["out"]
    kind = case["kind"]
    if kind == "evolve":
        g.step(case["steps"])
        return out.read(g)
    if kind == "method":
        for _ in range(case["steps"]):
            g.stepInit()
            for fin in (g.K1Finalize, g.K2Finalize, g.K3Finalize, g.K4Finalize):
                g.RKEvolve()
                fin()
        return out.read(g)
    if kind == "batch":
        g.step(case["steps"])
        return [o.read(m) for o, m in zip(out, g.members)]
    if kind == "output":
        c = g.setConstraintCalcs()
        # A and S measure the rounding of the normalisation here: no numbers to compare
        res = {k: np.array(c[k]) for k in ("H", "M", "G")}
        res.update(out.read(g, lambda f: f + "_a"))
        res["strip"] = g.strip("DIFFphi_a", 1, 3, 5)
        res["stats"] = np.array([g.field_stats(f) for f in ("DIFFphi_a", "DIFFK_a")])
        res["spec_phi"] = g.power_spectrum("DIFFphi_a")
        res["spec_rho"] = g.power_spectrum("DIFFr_a")
        return res
    if kind == "svt":
        viols = g.bardeen(0.1, True, 0.3)
        res = out.read(g, lambda f: "Bardeen_" + f)
        res["viols"] = viols
        return res
    c, _ = g.ics_static_dust(state["modes"], 1e-2)
    res = out.read(g, lambda f: f + ("_a" if f == "DIFFD" else "_p"))
    res["shift"] = c
    return res


# ------------------------------------------------------------------- work --
def _flops(case):
    """Operations of one right-hand side and update at a point, in round numbers: per differentiated field 9
    derivatives of 2R (first, second) and 4R (mixed) neighbours, then the BSSN algebra."""
    R = case["order"] // 2
    return 8 * 3 * (4 * R + 4 * R + 8 * R) + 4 * 3 * 4 * R + 1300


def work(case):
    kind = case["kind"]
    w = 8 if case["precision"] == "fp64" else 4
    if kind in ("evolve", "method"):
        pts = case["nx"] * case["ny"] * case["nz"]
        F = 17 + (case["lapse"] != "Static") + 4 * (case["matter"] == "dust") + 7 * (case["shift"] != "none")
        # per stage the stencil input and the step's start are read and the new state is written
        per = (2 + 3 + 3 + 3) * F * w + 4 * w * (case["matter"] == "static")
        return dict(bytes=float(pts) * (case["steps"] * per + 2 * w * len(_kept(case))),
                    flops=float(pts) * case["steps"] * 4 * _flops(case))
    if kind == "batch":
        pts = sum(n ** 3 for n in _members(case))
        return dict(bytes=float(pts) * (case["steps"] * (11 * 17 + 4) * w + 2 * 3 * w),
                    flops=float(pts) * case["steps"] * 4 * _flops(case))
    if kind == "output":
        pts = case["nx"] * case["ny"] * case["nz"]
        fft = 2.5 * math.log2(pts)
        return dict(bytes=float(pts) * (19 * w + 2 * 8 + 2 * 8 + 3 * 8), flops=float(pts) * (_flops(case) + 400 + 2 * fft))
    if kind == "svt":
        pts = case["nx"] * case["ny"] * case["nz"]
        fft = 2.5 * math.log2(pts)
        return dict(bytes=float(pts) * (19 * w + 5 * 8 + 14 * 2 * 8), flops=float(pts) * (2 * _flops(case) + 28 * fft))
    pts = case["n"] ** 3
    fft = 2.5 * math.log2(pts)
    return dict(bytes=float(pts) * (16 + 10 * 4 * 8 + 2 * 8), flops=float(pts) * 10 * (2 * fft + 20))


# ---------------------------------------------------------- 64-bit results --
C1 = {2: [1 / 2], 4: [2 / 3, -1 / 12], 6: [3 / 4, -3 / 20, 1 / 60], 8: [4 / 5, -1 / 5, 4 / 105, -1 / 280]}
C2 = {2: [-2.0, 1.0], 4: [-5 / 2, 4 / 3, -1 / 12], 6: [-49 / 18, 3 / 2, -3 / 20, 1 / 90],
      8: [-205 / 72, 8 / 5, -1 / 5, 8 / 315, -1 / 560]}
CM = {2: [1 / 4], 4: [1 / 3, -1 / 48], 6: [135 / 360, -13.5 / 360, 1 / 360], 8: [2 / 5, -1 / 20, 2 / 315, -1 / 2240]}
KO = {2: [6.0, -4.0, 1.0], 8: [-252.0, 210.0, -120.0, 45.0, -10.0, 1.0]}


class _Grid:
    def __init__(self, case):
        self.order, self.i1 = case["order"], float(case["nx"])

    def at(self, f, a, m):
        return torch.roll(f, -m, dims=a)

    def d1(self, f, a):
        return sum(c * (self.at(f, a, m) - self.at(f, a, -m)) for m, c in enumerate(C1[self.order], 1)) * self.i1

    def dd(self, f, a, b):
        if a == b:
            c = C2[self.order]
            s = c[0] * f
            for m in range(1, len(c)):
                s = s + c[m] * (self.at(f, a, m) + self.at(f, a, -m))
            return s * self.i1 ** 2
        s = 0
        for m, c in enumerate(CM[self.order], 1):
            p, q = self.at(f, a, m), self.at(f, a, -m)
            s = s + c * (self.at(p, b, m) - self.at(p, b, -m) - self.at(q, b, m) + self.at(q, b, -m))
        return s * self.i1 ** 2

    def ko(self, f, ko):
        if not ko or self.order not in KO:
            return 0.0
        w = KO[self.order]
        s = 3 * w[0] * f
        for m in range(1, len(w)):
            for a in range(3):
                s = s + w[m] * (self.at(f, a, m) + self.at(f, a, -m))
        return s * (ko / 64 if self.order == 2 else -ko / 1024) * self.i1

    def up(self, f, a, v):
        """The lopsided advection v d_a f (orders 2 and 4; zero at the others)."""
        at, dx = (lambda m: self.at(f, a, m)), 1.0 / self.i1
        if self.order == 2:
            fw = (-0.5 * at(2) + 2 * at(1) - 1.5 * f) / dx - 0.5 * (2 * f - 5 * at(1) + 4 * at(2) - at(3)) / dx
            bw = (0.5 * at(-2) - 2 * at(-1) + 1.5 * f) / dx + 0.5 * (2 * f - 5 * at(-1) + 4 * at(-2) - at(-3)) / dx
        elif self.order == 4:
            fw = (at(3) / 12 - 0.5 * at(2) + 1.5 * at(1) - 5 / 6 * f - 0.25 * at(-1)) / dx
            bw = (-at(-3) / 12 + 0.5 * at(-2) - 1.5 * at(-1) + 5 / 6 * f + 0.25 * at(1)) / dx
        else:
            return torch.zeros_like(f)
        return v * torch.where(v > 0, fw, bw)


def _normalised(s):
    """det(gamma) = 1 and A_ij trace free."""
    g = [s[m] for m in MET]
    g11, g12, g13, g22, g23, g33 = g
    x = -(g11 + g22 + g33 - g12 ** 2 - g13 ** 2 - g23 ** 2 + g11 * g22 + g11 * g33 + g22 * g33 - g23 ** 2 * g11 -
          g13 ** 2 * g22 - g12 ** 2 * g33 + 2 * g12 * g13 * g23 + g11 * g22 * g33)
    t = -torch.expm1(torch.log1p(-x) / 3)
    o = dict(s)
    for (a, b), m in zip(SYM, MET):
        o[m] = (s[m] + (t if a == b else 0)) / (1 - t)
    gi = _inverse([o[m] for m in MET])
    tr = sum((1 if a == b else 2) * gi[_sy(a, b)] * s[m] for (a, b), m in zip(SYM, AIJ))
    for (a, b), m, gm in zip(SYM, AIJ, MET):
        o[m] = (s[m] - (float(a == b) + o[gm]) * tr / 3) / (1 - t)
    return o


def _inverse(g):
    g11, g12, g13, g22, g23, g33 = g
    return [1 + g22 + g33 - g23 ** 2 + g22 * g33, g13 * g23 - g12 * (1 + g33), g12 * g23 - g13 * (1 + g22),
            1 + g11 + g33 - g13 ** 2 + g11 * g33, g12 * g13 - g23 * (1 + g11), 1 + g11 + g22 - g12 ** 2 + g11 * g22]


class _Frw:
    """RK4 of the background: phi, K and the fluids, stage by stage."""

    def __init__(self, frw):
        self.y0 = [frw["phi"], frw["K"]] + [r for r, _ in frw["fluids"]]
        self.w = [w for _, w in frw["fluids"]]
        self.y, self.k = list(self.y0), []

    def rho(self):
        return sum(self.y[2:])

    def S(self):
        return sum(3 * r * w for r, w in zip(self.y[2:], self.w))

    def stage(self, n, h):
        p, K, r = self.y[0], self.y[1], self.y[2:]
        src = sum(4 * PI * x * (1 + 3 * w) for x, w in zip(r, self.w))
        self.k.append([-K / 6, K * K / 3 + src] + [K * x * (1 + w) for x, w in zip(r, self.w)])
        if n < 4:
            c = h if n == 3 else h / 2
            self.y = [a + c * b for a, b in zip(self.y0, self.k[-1])]
        else:
            self.y0 = [a + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4) for a, k1, k2, k3, k4 in zip(self.y0, *self.k)]
            self.y, self.k = list(self.y0), []


def _geometry(G, s, frw):
    """Derivatives and curvature the right-hand side and the constraints share."""
    q = {}
    g = [s[m] for m in MET]
    gi = _inverse(g)
    q["gi"], q["GI"] = gi, lambda a, b: gi[_sy(a, b)]
    GM = q["GM"] = lambda a, b: g[_sy(a, b)] + float(a == b)
    GI = q["GI"]
    dg = [[G.d1(x, a) for x in g] for a in range(3)]
    q["dphi"] = dphi = [G.d1(s["DIFFphi"], a) for a in range(3)]
    q["dK"] = [G.d1(s["DIFFK"], a) for a in range(3)]
    q["GL"] = GL = [[0.5 * (dg[b][_sy(c, i)] + dg[c][_sy(b, i)] - dg[i][_sy(b, c)]) for b, c in SYM] for i in range(3)]
    q["Gam"] = Gm = [[sum(GI(i, m) * GL[m][t] for m in range(3)) for t in range(6)] for i in range(3)]
    q["Gd"] = Gd = [sum((1 if a == b else 2) * gi[t] * Gm[i][t] for t, (a, b) in enumerate(SYM)) for i in range(3)]
    q["dg"] = dg
    phi = q["phi"] = s["DIFFphi"] + frw.y[0]
    q["em4"], q["e4"] = torch.exp(-4 * phi), torch.exp(4 * phi)
    DD = [G.dd(s["DIFFphi"], a, b) - sum(Gm[m][t] * dphi[m] for m in range(3)) for t, (a, b) in enumerate(SYM)]
    ex = sum((1 if a == b else 2) * gi[t] * (DD[t] + 2 * dphi[a] * dphi[b]) for t, (a, b) in enumerate(SYM))
    dG = [[G.d1(s[f], a) for f in GAM] for a in range(3)]  # dG[a][k] = d_a Gamma^k
    X = [[[sum(GI(m, l) * Gm[k][_sy(l, i)] for l in range(3)) for m in range(3)] for i in range(3)] for k in range(3)]

    def Z(i, j):
        return sum(X[k][i][m] * (GL[j][_sy(k, m)] + 0.5 * GL[k][_sy(m, j)]) for k in range(3) for m in range(3))

    ric = []
    for t, (a, b) in enumerate(SYM):
        lap = sum((1 if c == d else 2) * gi[u] * G.dd(g[t], c, d) for u, (c, d) in enumerate(SYM))
        t2 = sum(GM(k, a) * dG[b][k] + GM(k, b) * dG[a][k] for k in range(3))
        t3 = sum(Gd[k] * (GL[a][_sy(b, k)] + GL[b][_sy(a, k)]) for k in range(3))
        ric.append(-0.5 * lap + 0.5 * t2 + 0.5 * t3 + Z(a, b) + Z(b, a) -
                   2 * (DD[t] - 2 * dphi[a] * dphi[b] + GM(a, b) * ex))
    q["ric"] = ric
    q["ricci"] = q["em4"] * sum((1 if a == b else 2) * ric[t] * gi[t] for t, (a, b) in enumerate(SYM))
    A = [s[m] for m in AIJ]
    q["A"] = AM = lambda a, b: A[_sy(a, b)]
    q["Ac"] = Ac = [sum(GI(a, p) * GI(b, r) * AM(p, r) for p in range(3) for r in range(3)) for a, b in SYM]
    q["AA"] = sum((1 if a == b else 2) * Ac[t] * A[t] for t, (a, b) in enumerate(SYM))
    return q


def _rhs(G, case, s, frw, DIFFD, lag):
    """d_t of every evolved field at state s; `lag`: the state (with its FRW phi) the dust sources' W, detg, g_ij are of."""
    q = _geometry(G, s, frw)
    GI, GM, AM, gi = q["GI"], q["GM"], q["A"], q["gi"]
    phiF, KF, rF, SF = frw.y[0], frw.y[1], frw.rho(), frw.S()
    dphi, dK, Gm, Ac, em4, e4 = q["dphi"], q["dK"], q["Gam"], q["Ac"], q["em4"], q["e4"]
    al = 1 + s["DIFFalpha"]
    k, K = s["DIFFK"], s["DIFFK"] + KF
    live = case["lapse"] != "Static"
    dal = [G.d1(s["DIFFalpha"], a) for a in range(3)] if live else [0.0] * 3
    r, S, Si, STF, out = 0.0, 0.0, [0.0] * 3, [0.0] * 6, {}
    if case["matter"] == "static":
        r = torch.exp(-6 * q["phi"]) * DIFFD + rF * torch.expm1(-6 * s["DIFFphi"])
    if case["matter"] == "dust":
        D, Sd = s["dust_D"], [s[f] for f in DUST[1:]]

        def lorentz(st, pF):
            p = st["DIFFphi"] + pF
            h = _inverse([st[m] for m in MET])
            ss = sum((1 if a == b else 2) * h[t] * st[DUST[1 + a]] * st[DUST[1 + b]] for t, (a, b) in enumerate(SYM))
            return torch.sqrt(1 + torch.exp(-4 * p) * ss / st["dust_D"] ** 2), torch.exp(6 * p), torch.exp(4 * p)

        W, e6, _ = lorentz(s, phiF)
        v = [em4 / e6 * sum(GI(i, j) * Sd[j] for j in range(3)) for i in range(3)]
        ls, lp = lag if lag else (s, phiF)
        Wl, detg, e4l = lorentz(ls, lp)
        r = Wl * D / detg
        S = D / detg * (Wl * Wl - 1) / Wl
        Si = [x / detg for x in Sd]
        STF = [Sd[a] * Sd[b] / Wl / D / detg - e4l * (ls[m] + float(a == b)) * S / 3 for (a, b), m in zip(SYM, MET)]
        r, S = r - rF + LAMBDA, S - SF - 3 * LAMBDA
        out["dust_D"] = sum(G.d1(al * D * v[i], i) for i in range(3))
        for j in range(3):
            acc = sum((1 if a == b else 2) * v[a] * v[b] * (4 * dphi[j] * GM(a, b) + q["dg"][j][t])
                      for t, (a, b) in enumerate(SYM))
            out[DUST[1 + j]] = sum(G.d1(al * Sd[j] * v[i], i) for i in range(3)) + 0.5 * al * W * D * e4 * acc - W * D * dal[j]
    DDa, tr = [0.0] * 6, 0.0
    if live:
        gild = [sum(GI(i, j) * dphi[j] for j in range(3)) for i in range(3)]
        DDa = [G.dd(s["DIFFalpha"], a, b) - sum((Gm[m][t] + 2 * (float(m == a) * dphi[b] + float(m == b) * dphi[a] -
                                                                   GM(a, b) * gild[m])) * dal[m] for m in range(3))
               for t, (a, b) in enumerate(SYM)]
        tr = sum((1 if a == b else 2) * gi[t] * DDa[t] for t, (a, b) in enumerate(SYM))
        DDa = [DDa[t] - GM(a, b) * tr / 3 for t, (a, b) in enumerate(SYM)]
        tr = tr * em4
    for t, (a, b) in enumerate(SYM):
        out[MET[t]] = -2 * al * s[AIJ[t]]
        AA = sum(AM(m, a) * GI(m, n) * AM(n, b) for m in range(3) for n in range(3))
        TF = q["ric"][t] - e4 * GM(a, b) * q["ricci"] / 3
        out[AIJ[t]] = em4 * (al * (TF - 8 * PI * STF[t]) - DDa[t]) + al * (K * s[AIJ[t]] - 2 * AA)
    for i in range(3):
        sec = sum((1 if a == b else 2) * Gm[i][t] * Ac[t] for t, (a, b) in enumerate(SYM)) + \
            6 * sum(Ac[_sy(i, j)] * dphi[j] for j in range(3))
        out[GAM[i]] = -2 * sum(Ac[_sy(i, j)] * dal[j] for j in range(3)) + 2 * al * (
            sec - 2 / 3 * sum(GI(i, j) * dK[j] for j in range(3)) - 8 * PI * sum(GI(i, j) * Si[j] for j in range(3)))
    out["DIFFK"] = -tr + al * (k * (k + 2 * KF) / 3 + q["AA"]) + 4 * PI * al * (r + S) + 4 * PI * s["DIFFalpha"] * (rF + SF)
    out["DIFFphi"] = -(al * k + s["DIFFalpha"] * KF) / 6
    out["DIFFalpha"] = torch.zeros_like(k)
    if case["lapse"] == "Harmonic":
        out["DIFFalpha"] = -al * K
    elif case["lapse"] == "OnePlusLog":
        w = torch.exp(6 * q["phi"])
        out["DIFFalpha"] = -2 * al * (K - (w * k).sum() / w.sum())
    for f in MET + ["DIFFphi", "DIFFK", "DIFFalpha"] + AIJ + GAM:
        out[f] = out[f] - G.ko(s[f], case["ko"])
    if case["shift"] != "none":
        be = [s[f] for f in BETA]
        db = [[G.d1(b, j) for b in be] for j in range(3)]  # db[j][m] = d_j beta^m
        div = db[0][0] + db[1][1] + db[2][2]
        adv = lambda f: sum(G.up(s[f], a, be[a]) for a in range(3))  # noqa: E731
        for f in MET + ["DIFFphi", "DIFFK", "DIFFalpha"] + AIJ + GAM:
            out[f] = out[f] + adv(f)
        for t, (a, b) in enumerate(SYM):
            out[MET[t]] = out[MET[t]] + sum(GM(a, m) * db[b][m] + GM(b, m) * db[a][m] for m in range(3)) - 2 / 3 * GM(a, b) * div
            out[AIJ[t]] = out[AIJ[t]] + sum(AM(a, m) * db[b][m] + AM(b, m) * db[a][m] for m in range(3)) - 2 / 3 * AM(a, b) * div
        out["DIFFphi"] = out["DIFFphi"] + div / 6
        hess = [[G.dd(b, c, d) for c, d in SYM] for b in be]
        for i in range(3):
            lap = sum((1 if c == d else 2) * gi[u] * hess[i][u] for u, (c, d) in enumerate(SYM))
            gd = sum(GI(i, j) * sum(hess[m][_sy(j, m)] for m in range(3)) for j in range(3))
            out[GAM[i]] = out[GAM[i]] - sum(q["Gd"][j] * db[j][i] for j in range(3)) + 2 / 3 * q["Gd"][i] * div + lap + gd / 3
            out[BETA[i]] = s[AUXB[i]] - 0.0
            out[AUXB[i]] = 0.75 * out[GAM[i]] - 1.0 * s[AUXB[i]]
        if case["lapse"] == "OnePlusLog":
            out["DIFFalpha"] = out["DIFFalpha"] + sum(be[a] * dal[a] for a in range(3))
    return out


def _evolve(case, seed):
    fields, bg = _start(case, seed)
    shape, h, G, frw = _shape(case), 0.1 / case["nx"], _Grid(case), _Frw(bg)
    DIFFD = fields.pop("DIFFD", None)
    names = FIELDS + ["DIFFalpha"] + (BETA + AUXB if case["shift"] != "none" else []) + (DUST if case["matter"] == "dust" else [])
    p = {f: fields[f].clone() if f in fields else torch.zeros(shape, device="cuda", dtype=torch.float64) for f in names}
    for _ in range(case["steps"]):
        a, acc, lag = _normalised(p), None, None
        for n in (1, 2, 3, 4):
            d = _rhs(G, case, a, frw, DIFFD, lag)
            lag = (a, frw.y[0])
            frw.stage(n, h)
            w = h / 6 if n in (1, 4) else h / 3
            acc = {f: w * d[f] if acc is None else acc[f] + w * d[f] for f in names}
            if n < 4:
                a = {f: p[f] + (h if n == 3 else h / 2) * d[f] for f in names}
        p = {f: p[f] + acc[f] for f in names}
    return p


def _strip(x, n1, n2):
    return x[:, n1, n2]


def _spectrum(f):
    nx, ny, nz = f.shape
    kx, ky, kz = _lattice(f.shape)
    w = torch.where((kz > 0) & (kz < nz // 2), 2.0, 1.0).double()
    b = torch.sqrt(kx * kx + ky * ky + kz * kz).long().reshape(-1)
    nb = int(math.sqrt(nx * nx + ny * ny + nz * nz) / 2.0) + 1
    s = torch.zeros(nb, device="cuda", dtype=torch.float64).index_add_(0, b, (w * torch.fft.rfftn(f).abs() ** 2).reshape(-1))
    c = torch.zeros_like(s).index_add_(0, b, w.reshape(-1))
    return torch.where(c > 0, s / torch.where(c > 0, c, torch.ones_like(c)), torch.zeros_like(s))


def _stats(val, scale, dx, l2):
    n, sc = val.numel(), val / scale
    o = [val.mean(), val.std(), val.abs().max(), scale.sum(), sc.mean(), sc.std(), sc.abs().max()]
    o += [torch.sqrt((val * val).sum() * dx ** 3)] if l2 else []
    return torch.stack(o) if n else None


def _output(case, seed):
    case = dict(case, matter="static", lapse="Harmonic", shift="none", ko=0.0)
    f = _general(case, seed)
    D = f.pop("DIFFD")
    s, G, frw = _normalised(f), _Grid(case), _Frw(dict(phi=0.0, K=0.0, fluids=[]))
    q = _geometry(G, s, frw)
    GI, AM, gi, dphi = q["GI"], q["A"], q["gi"], q["dphi"]
    dx, K, p = 1.0 / case["nx"], s["DIFFK"], q["phi"]
    r = torch.exp(-6 * p) * D
    H = -torch.exp(5 * p) / 8 * (q["ricci"] + 2 / 3 * K * K - q["AA"] - 16 * PI * r)
    Hs = torch.exp(5 * p) / 8 * torch.sqrt(q["ricci"] ** 2 + q["AA"] ** 2 + (2 / 3 * K * K) ** 2 + (16 * PI * r) ** 2)
    M2, Ms2, G2, Gs2 = 0, 0, 0, 0
    for i in range(3):
        dA = [[G.d1(s[AIJ[_sy(m, i)]], n) for m in range(3)] for n in range(3)]
        t6 = sum(GI(m, n) * AM(m, i) * dphi[n] for m in range(3) for n in range(3))
        td = sum(GI(m, n) * dA[n][m] for m in range(3) for n in range(3)) - sum(q["Gd"][m] * AM(m, i) for m in range(3)) - \
            sum(q["GL"][m][_sy(n, i)] * q["Ac"][_sy(m, n)] for m in range(3) for n in range(3))
        e6 = torch.exp(6 * p)
        M2 = M2 + (e6 * (-2 / 3 * q["dK"][i] + 6 * t6 + td)) ** 2
        Ms2 = Ms2 + (e6 * ((2 / 3 * q["dK"][i]).abs() + 6 * t6.abs() + td.abs())) ** 2
        Gi = q["Gam"][i]
        G2 = G2 + (s[GAM[i]] - q["Gd"][i]) ** 2
        dia = gi[0] * Gi[0] - gi[3] * Gi[3] - gi[5] * Gi[5] - 2 * (gi[1] * Gi[1] + gi[2] * Gi[2] + gi[4] * Gi[4])
        Gs2 = Gs2 + (s[GAM[i]].abs() + dia.abs()) ** 2
    res = {"H": _stats(H, Hs, dx, True), "M": _stats(torch.sqrt(M2), torch.sqrt(Ms2), dx, True),
           "G": _stats(torch.sqrt(G2), torch.sqrt(Gs2), dx, False), "ricci": q["ricci"], "AijAij": q["AA"]}
    # a context that has not stepped reads _a as _p
    res["strip"] = _strip(f["DIFFphi"], 3, 5)
    w = torch.exp(6 * f["DIFFphi"])
    rows = []
    for x in (f["DIFFphi"], f["DIFFK"]):
        vol = w.mean()
        avg = (w * x).mean() / vol
        rows.append(torch.stack([avg, torch.sqrt((w * (avg - x) ** 2).sum() / (x.numel() - 1) / vol), vol]))
    res["stats"] = torch.stack(rows)
    res["spec_phi"], res["spec_rho"] = _spectrum(f["DIFFphi"]), _spectrum(r)
    return res


def _svt(case, seed):
    case = dict(case, matter="static", lapse="Harmonic", shift="none", ko=0.0)
    f = _general(case, seed)
    D = f.pop("DIFFD")
    s, G = _normalised(f), _Grid(case)
    c = _rhs(G, case, s, _Frw(dict(phi=0.0, K=0.0, fluids=[])), D, None)
    OL, t = 0.3, 0.1
    so = math.sqrt(OL)
    a = (math.cosh(1.5 * so * t) + math.sinh(1.5 * so * t) / so) ** (2 / 3)
    Hb = math.sqrt((1 - OL) * a ** -3 + OL)
    ad, add = Hb * a, a * Hb * Hb - (1 - OL) * 1.5 / a / a
    kx, ky, kz = _lattice(_shape(case))
    k2 = (kx * kx + ky * ky + kz * kz) * (2 * PI) ** 2

    def inv(x):
        X = torch.fft.rfftn(x) / -torch.where(k2 > 0, k2, torch.ones_like(k2))
        X[0, 0, 0] = 0
        return torch.fft.irfftn(X, s=_shape(case))

    al, phi, dt, K = 1 + s["DIFFalpha"], s["DIFFphi"], c["DIFFphi"], s["DIFFK"]
    e4 = torch.exp(4 * phi)
    d2p = -(c["DIFFalpha"] * K + al * c["DIFFK"]) / 6
    h, dh, ddh = [], [], []
    for (i, j), m, n in zip(SYM, MET, AIJ):
        u, g = float(i == j), s[m] + float(i == j)
        d2g = -2 * c["DIFFalpha"] * s[n] - 2 * al * c[n]
        h.append(e4 * g - u * a * a)
        dh.append(e4 * (4 * dt * g + c[m]) - u * 2 * a * ad)
        ddh.append(e4 * (16 * dt * dt * g + 8 * dt * c[m] + 4 * d2p * g + d2g) - u * 2 * (ad * ad + a * add))
    tr = [x[0] + x[3] + x[5] for x in (h, dh, ddh)]
    E = al * al - 1
    dd = [inv(sum((1 if i == j else 2) * G.dd(x[u], i, j) for u, (i, j) in enumerate(SYM))) for x in (h, dh, ddh)]
    A = (tr[0] - dd[0]) / a / a / 2
    dA = -2 * A * Hb + (tr[1] - dd[1]) / a / a / 2
    ddA = -2 * A * (Hb * Hb + add / a) - 4 * Hb * dA + (tr[2] - dd[2]) / a / a / 2
    m = [x.mean() for x in tr]
    A = A + m[0] / 3 / a / a - A.mean()
    dA = dA + m[1] / 3 / a / a - 2 * m[0] * ad / 3 / a ** 3 - dA.mean()
    ddA = ddA + m[2] / 3 / a / a - 2 * ad * m[1] / 3 / a ** 3 + 6 * m[0] * ad * ad / 3 / a ** 4 - \
        2 * m[0] * add / 3 / a ** 3 - 2 * m[1] * ad / 3 / a ** 3 - ddA.mean()
    B = inv(tr[0] / a / a - 3 * A)
    dB = inv(tr[1] / a / a - 2 / a ** 3 * ad * tr[0] - 3 * dA)
    ddB = inv(tr[2] / a / a - 4 / a ** 3 * ad * tr[1] - 2 / a ** 3 * add * tr[0] + 6 / a ** 4 * ad * ad * tr[0] - 3 * ddA)
    Psi = -0.5 * (A - Hb * a * a * dB)
    Phi = 0.5 * (E - 2 * a * ad * dB - a * a * ddB)

    def vec(x, X, i):
        o = [j for j in range(3) if j != i]
        return sum(G.d1(x[_sy(i, j)], j) - G.d1(x[_sy(j, j)], i) for j in o) / a / a + X

    raw = [vec(h, 2 * G.d1(A, i), i) for i in range(3)]
    dC = [inv(vec(dh, 2 * G.d1(dA, i), i) - 2 * Hb * (raw[i] - 2 * G.d1(A, i))) for i in range(3)]
    Cv = inv(raw[0])
    V = torch.sqrt(sum((a * x) ** 2 for x in dC))
    D11 = h[0] / a / a - A - G.dd(B, 0, 0) - 2 * G.d1(Cv, 0)

    def ab(x):
        return sum(G.dd(x, i, j).abs() for i, j in SYM)

    lv = E + A - a * a * ddB - 3 * a * ad * dB
    mag = torch.sqrt(E * E + A * A + (a * a * ddB) ** 2 + (3 * a * ad * dB) ** 2)
    dmag = ab(E) + ab(A) + a * a * ab(ddB) + 3 * a * ad * ab(dB)
    dv = ab(lv)
    w = torch.exp(6 * phi)
    cav = lambda x: (w * x).sum() / w.sum()  # noqa: E731
    am, Km = 1 + cav(s["DIFFalpha"]), cav(K)
    v = [dv.mean() / dmag.mean(), dv.std() / dmag.mean(), dv.max() / dmag.mean(), dv.max(), lv.mean() / mag.mean(),
         lv.std() / mag.mean(), lv.max() / mag.mean(), lv.max(), 1 - a / torch.exp(2 * cav(phi)),
         1 + Hb * 3 / (a * am * Km), 1 - add / (Hb * ad + 2 * a * cav(d2p)), 1 - a / torch.exp(2 * phi.mean()),
         1 + Hb * 3 / (a * am * K.mean()), 1 - add / (Hb * ad + 2 * a * d2p.mean()), V.mean(), V.std(), V.max()]
    return {"Phi": Phi, "Psi": Psi, "B": B, "C1": Cv, "D11": D11, "viols": torch.stack(v)}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("evolve", "method"):
        p = _evolve(case, seed)
        return {f: p[f] for f in _kept(case)}
    if kind == "batch":
        res = []
        for r, n in enumerate(_members(case)):
            p = _evolve(_member(case, n), seed * 64 + r)
            res.append({f: p[f] for f in ("DIFFphi", "DIFFK", "A12")})
        return res
    if kind == "output":
        return _output(case, seed)
    if kind == "svt":
        return _svt(case, seed)
    n = case["n"]
    phi, D, c = _solve(_modes((n, n, n), seed), (n, n, n), 1e-2, 1.0 / n)
    return {"DIFFphi": phi, "DIFFD": D - RHO_BAR, "shift": c}
