"""Timed workloads of the framework, through its public entry points.

`listed()` names the workloads, `draw(rng)` gives more of the same ranges,
`prepare` / `run` set one up and take one pass through it, `work` is the data
and arithmetic a pass cannot do without, and `exact` is what a pass returns,
computed in 64 bits with plain torch.

Families (the "kind" of a case):
  mhd      Integrator.run: `steps` whole MHD steps of one grid (CFL, four RK
           stages, the artificial-viscosity sweeps, ghost fills), 2D or 3D
  ensemble Ensemble.step: a captured hipGraph of `steps` steps over many
           independent 2D Kelvin-Helmholtz runs of uneven size
  rmhd     RadiativeMHD.step_plain: an RT solve, Q_rad and the heated MHD step
           of the gravity-stratified radiative box
  rt       RT: opacity and source from the fields, a solve from zero
           intensities to the tolerance, Q_rad and the intensities
  slab     BottomSlabRT.apply: the two-iteration RT solve of a thin slab at
           the bottom of a box, which the learned stepping runs at every step
  predict  ColumnSurrogate.predict: features, network and Q_rad of a whole box
  fit      ColumnSurrogate.fit: epochs of forward, backward and Adam, then the
           trained weights
"""
import ctypes as C
import math

import numpy as np
import torch

from miso_amd import ensemble, hip, mhd, rmhd, rt, surrogate

DEV = "cuda:0"
RO, VX, VY, VZ, BX, BY, BZ, EI, PH = range(9)
# mirror signs: the velocity and field component along the axis flip
SIGNS = tuple(tuple(-1 if f in (VX + a, BX + a) else 1 for f in range(9)) for a in range(3))
HIDDEN, HIDDEN_LAYERS, FEATURES, LAPLACIAN_STRIDE = 256, 3, 4, 4


def listed():
    return [
        # the smallest calls: the 2D Orszag-Tang vortex of the parity runs,
        # launch-bound, ten steps a call
        dict(name="vortex_256_f64", kind="mhd", nx=256, ny=256, nz=1, dtype="f64", ic="vortex",
             bc="periodic", steps=10),
        # an ordinary 2D run with odd sizes, FP32, walls in y
        dict(name="shear_1131x757_f32", kind="mhd", nx=1131, ny=757, nz=1, dtype="f32",
             ic="shear", bc="mirror_y", steps=4),
        # a small 3D box: too few cells to fill the chip
        dict(name="turbulence_64_f64", kind="mhd", nx=64, ny=64, nz=64, dtype="f64",
             ic="turbulence", bc="periodic", steps=4),
        # an ordinary 3D box, no size a multiple of a tile, walls in z
        dict(name="turbulence_205x131x93_f64", kind="mhd", nx=205, ny=131, nz=93, dtype="f64",
             ic="turbulence", bc="mirror_z", steps=2),
        # the headline box in both precisions
        dict(name="turbulence_512_f64", kind="mhd", nx=512, ny=512, nz=512, dtype="f64",
             ic="turbulence", bc="periodic", steps=2),
        dict(name="turbulence_512_f32", kind="mhd", nx=512, ny=512, nz=512, dtype="f32",
             ic="turbulence", bc="periodic", steps=2),
        # the batched ensemble: 64 runs of 128^2 ... 1024^2, FP32
        dict(name="ensemble_64_f32", kind="ensemble", runs=64, pick=7, steps=4),
        # radiative MHD with the plain solver on every step
        dict(name="radiative_step_256", kind="rmhd", nx=256, ny=256, nz=256),
        # a cold RT solve of an ordinary, odd-sized box
        dict(name="rt_solve_211x150x187", kind="rt", nx=211, ny=150, nz=187),
        # the learned stepping's three parts: the slab solve, the network on a
        # whole box, and its training
        dict(name="rt_slab_384x27", kind="slab", nx=384, ny=384, nz=384, layers=23, buffer=4),
        dict(name="predict_384", kind="predict", nx=384, ny=384, nz=384),
        dict(name="fit_384_batch1024", kind="fit", nz=384, columns=16384, batch=1024, epochs=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mhd", "mhd", "mhd", "mhd", "ensemble", "rmhd", "rt", "slab", "predict",
                       "fit"])
    if kind == "mhd":
        dtype = rng.choice(["f64", "f32"])
        if rng.random() < 0.4:
            ic = rng.choice(["vortex", "shear"])
            return dict(kind=kind, nx=_log(rng, 96, 1600), ny=_log(rng, 96, 1600), nz=1,
                        dtype=dtype, ic=ic, bc="mirror_y" if ic == "shear" else "periodic",
                        steps=rng.choice([2, 4, 10]))
        return dict(kind=kind, nx=_log(rng, 40, 420), ny=_log(rng, 40, 420),
                    nz=_log(rng, 40, 420), dtype=dtype, ic="turbulence",
                    bc=rng.choice(["periodic", "periodic", "mirror_z"]), steps=2)
    if kind == "ensemble":
        return dict(kind=kind, runs=rng.randint(6, 60), pick=rng.randrange(1000),
                    steps=rng.choice([2, 4]))
    if kind in ("rmhd", "rt"):
        return dict(kind=kind, nx=_log(rng, 48, 230), ny=_log(rng, 48, 230),
                    nz=_log(rng, 64, 230))
    if kind == "slab":
        return dict(kind=kind, nx=rng.randint(96, 384), ny=rng.randint(96, 384),
                    nz=rng.randint(192, 384), layers=rng.randint(10, 26),
                    buffer=rng.randint(2, 5))
    if kind == "predict":
        return dict(kind=kind, nx=rng.randint(60, 384), ny=rng.randint(60, 384),
                    nz=32 * rng.randint(2, 12))
    return dict(kind=kind, nz=32 * rng.randint(3, 12), columns=_log(rng, 6000, 16384),
                batch=32 * rng.randint(4, 32), epochs=rng.randint(1, 3))


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _np_dtype(case):
    return np.float32 if case.get("dtype") == "f32" else np.float64


# ------------------------------------------------------------------ MHD runs
def _bounds(case):
    """Cubic cells, the longest axis of length one."""
    n = max(case["nx"], case["ny"], case["nz"])
    return tuple((0.0, case[a] / n if case[a] > 1 else 1.0) for a in ("nx", "ny", "nz"))


def _coords(case):
    """Cell centres with ghosts, each axis shaped for (k, j, i) arrays."""
    out = []
    for a, key in enumerate(("nx", "ny", "nz")):
        n, hi = case[key], _bounds(case)[a][1]
        m = 2 if n > 1 else 0
        x = (torch.arange(n + 2 * m, dtype=torch.float64, device=DEV) - m + 0.5) * (hi / n)
        out.append((x / hi if n > 1 else x * 0).reshape([-1 if 2 - a == d else 1
                                                          for d in range(3)]))
    return out


def _initial(case, seed):
    """(9, Kt, Jt, It) state, ghosts included, of one seeded initial condition."""
    rng = np.random.default_rng(seed)
    x, y, z = _coords(case)
    shape = (z.numel(), y.numel(), x.numel())
    q = torch.zeros((9,) + shape, dtype=torch.float64, device=DEV)
    tau = 2 * math.pi
    if case["ic"] == "vortex":  # Orszag-Tang, amplitudes near the usual ones
        a, b = rng.uniform(0.9, 1.1, 2)
        b0 = b / math.sqrt(4 * math.pi)
        q[RO] = 25 / (36 * math.pi)
        q[EI] = 5 / (12 * math.pi) / (2 / 3) / (25 / (36 * math.pi))
        q[VX] = -a * torch.sin(tau * y)
        q[VY] = a * torch.sin(tau * x)
        q[BX] = -b0 * torch.sin(tau * y)
        q[BY] = b0 * torch.sin(2 * tau * x)
    elif case["ic"] == "shear":  # Kelvin-Helmholtz layer, seeded perturbation
        t = torch.tanh((y - 0.5) / 0.02)
        q[RO] = 1.5 - 0.5 * t
        q[VX] = 0.5 * t
        q[VY] = 1e-3 * (2 * torch.rand(shape, generator=_gen(seed), dtype=torch.float64,
                                       device=DEV) - 1)
        q[BX] = rng.uniform(0.0, 0.2)
        q[EI] = 2.5 / (2 / 3) / q[RO]
    else:  # decaying turbulence: random modes, B of each mode normal to k
        q[RO] = 1.0
        q[EI] = 1.5
        for first, rms, solenoidal in ((VX, 0.5, False), (BX, 0.3, True)):
            for _ in range(6):
                k = rng.integers(-3, 4, 3).astype(float)
                k[0] += not k.any()
                amp = rng.normal(size=3)
                if solenoidal:  # normal to the wave vector of the box's extents
                    w = k / [hi for _, hi in _bounds(case)]
                    amp -= w * (amp @ w) / (w @ w)
                phase = torch.sin(tau * (k[0] * x + k[1] * y + k[2] * z) + rng.uniform(0, tau))
                for c in range(3):
                    q[first + c] += float(rms * amp[c] / math.sqrt(18.0)) * phase
    return q.to(torch.float32 if _np_dtype(case) is np.float32 else torch.float64)


def _bc(case):
    kinds = [True, True, True]
    if case["bc"] == "mirror_y":
        kinds[1] = False
    if case["bc"] == "mirror_z":
        kinds[2] = False
    return mhd.BoundaryCondition(tuple(kinds), SIGNS)


def _prepare_mhd(case, seed):
    grid = mhd.Grid(case["nx"], case["ny"], case["nz"], 2, bounds=_bounds(case),
                    dtype=_np_dtype(case), device=DEV)
    ctx = mhd.ExecContext(0)
    model = mhd.MHD(mhd.Config({"mhd": {"cfl_number": 0.4}}), grid, ctx, gm=5 / 3)
    model.qq.data.copy_(_initial(case, seed))
    bc = _bc(case)
    model.integrator.apply_boundary_condition(bc, model.qq)
    return dict(model=model, bc=bc, steps=case["steps"])


def _run_mhd(s):
    m = s["model"]
    dts = m.integrator.run(s["bc"], m.qq, s["steps"])
    return {"q": m.qq.data, "dt": dts}


class _Scheme:
    """The MHD step in plain torch, float64: 4th-order central differences,
    four RK stages, the limited artificial viscosity along x, y and z.  min
    and max in the limiter and the CFL condition narrow to float, as the
    scheme defines them."""

    def __init__(self, n, spacing, real, kinds, gm=5 / 3, cfl=0.4, grav=0.0, fixed=None):
        self.n, self.kinds, self.gm, self.cfl, self.grav, self.fixed = n, kinds, gm, cfl, grav, fixed
        self.m = [2 if k > 1 else 0 for k in n]
        d = [real(s) if k > 1 else real(1e30) for s, k in zip(spacing, n)]
        self.di = [float(real(1.0 / float(x))) if k > 1 else 0.0 for x, k in zip(d, n)]
        self.hmin = float(np.float32(min(float(x) for x in d)))

    def inner(self, f, but=None):
        for a in range(3):
            if a != but:
                f = f.narrow(f.dim() - 1 - a, self.m[a], self.n[a])
        return f

    def fill(self, q):
        for a in range(3):
            n, m = self.n[a], self.m[a]
            if n == 1:
                continue
            v = q.transpose(3 - a, 0)  # the axis first, fields in its place
            if self.kinds[a] == "periodic":
                v[:m] = v[n:n + m].clone()
                v[n + m:] = v[m:2 * m].clone()
            elif self.kinds[a] == "mirror":
                for f in range(9):
                    w = q[f].transpose(2 - a, 0)
                    w[:m] = SIGNS[a][f] * w[m:2 * m].flip(0)
                    w[n + m:] = SIGNS[a][f] * w[n:n + m].flip(0)
            else:
                v[:m] = self.fixed.transpose(3 - a, 0)[:m]
                v[n + m:] = self.fixed.transpose(3 - a, 0)[n + m:]
        return q

    def diff(self, f, a):
        f = self.inner(f, but=a)
        w = lambda o: f.narrow(2 - a, 2 + o, self.n[a])  # noqa: E731
        return (8 * (w(1) - w(-1)) - w(2) + w(-2)) * (self.di[a] / 12)

    def stage(self, orgn, argm, dt, ch2, damp):
        ro, v, b, ei, ph = argm[0], argm[1:4], argm[4:7], argm[7], argm[8]
        p4, p8 = 1 / (4 * math.pi), 1 / (8 * math.pi)
        pr = (self.gm - 1) * ro * ei
        bb = b[0] ** 2 + b[1] ** 2 + b[2] ** 2
        ht = ro * ei + pr + bb * p4 + 0.5 * ro * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
        vb = v[0] * b[0] + v[1] * b[1] + v[2] * b[2]
        pt = pr + bb * p8
        o = self.inner(orgn)
        d_ro = torch.zeros_like(o[0])
        d_m, d_b = torch.zeros_like(o[1:4]), torch.zeros_like(o[4:7])
        d_e, d_p = torch.zeros_like(o[0]), torch.zeros_like(o[0])
        for a in range(3):
            if self.n[a] == 1:
                continue
            d_ro -= self.diff(ro * v[a], a)
            for c in range(3):
                d_m[c] += self.diff(p4 * b[c] * b[a] - ro * v[c] * v[a], a)
                if c != a:
                    d_b[c] += self.diff(v[c] * b[a] - b[c] * v[a], a)
            d_m[a] -= self.diff(pt, a)
            d_b[a] -= self.diff(ph, a)
            d_e += self.diff(p4 * vb * b[a] - ht * v[a], a)
            d_p -= self.diff(b[a], a)
        if self.grav:
            d_m[2] -= self.grav * self.inner(ro)
        out = torch.empty_like(argm)
        r = self.inner(out)
        r[0] = o[0] + dt * d_ro
        r[1:4] = (o[0] * o[1:4] + dt * d_m) / r[0]
        r[4:7] = o[4:7] + dt * d_b
        r[8] = (o[8] + dt * ch2 * d_p) * damp
        e = o[0] * o[7] + 0.5 * o[0] * (o[1:4] ** 2).sum(0) + p8 * (o[4:7] ** 2).sum(0) + dt * d_e
        r[7] = (e - 0.5 * r[0] * (r[1:4] ** 2).sum(0) - p8 * (r[4:7] ** 2).sum(0)) / r[0]
        return self.fill(out)

    def speeds(self, q):
        return (torch.sqrt(self.gm * (self.gm - 1) * q[7]), torch.sqrt((q[1:4] ** 2).sum(0)),
                torch.sqrt((q[4:7] ** 2).sum(0) / q[0] / (4 * math.pi)))

    def cfl_dt(self, q):
        total = sum(self.speeds(self.inner(q)))
        return float((self.cfl * self.hmin / total).min().float())

    def sweep(self, q, cc, a, dt):
        n, dim = self.n[a], 2 - a
        p = self.inner(q, but=a)
        cc = self.inner(cc, but=a)
        at = lambda f, o, k: f.narrow(dim, o, k)  # noqa: E731
        cf = 0.5 * (at(cc, 1, n + 1) + at(cc, 2, n + 1))
        ro = p[0]
        out = torch.empty_like(q)
        r = self.inner(out)
        c0 = lambda f: at(f, 2, n)  # noqa: E731
        e = 0.0
        for f in range(9):
            v = p[f] if f in (RO, BX, BY, BZ, PH) else ro * p[f]
            up = at(v, 1, n + 3) - at(v, 0, n + 3)
            lo, hi = at(up, 0, n + 2), at(up, 1, n + 2)
            mid = 0.5 * (at(v, 2, n + 2) - at(v, 0, n + 2))
            big = torch.maximum(torch.maximum(lo.float(), hi.float()), mid.float())
            small = torch.minimum(torch.minimum(lo.float(), hi.float()), mid.float())
            s = (big.clamp(max=0.0) + small.clamp(min=0.0)).double()
            dv = at(v, 2, n + 1) - at(v, 1, n + 1)
            jump = dv - 0.5 * (at(s, 0, n + 1) + at(s, 1, n + 1))
            den = torch.copysign(dv.abs().float().clamp(min=1e-20).double(), dv)
            ra = (jump / den).float().clamp(max=1.0).double()
            pp = (0.5 + torch.copysign(torch.full_like(ra, 0.5), ra)) * ra.clamp(min=0.0)
            flux = -0.5 * cf * pp * jump
            df = (at(flux, 1, n) - at(flux, 0, n)) * (self.di[a] * dt)
            if f in (VX, VY, VZ):
                r[f] = (c0(v) - df) / r[0]
            elif f == EI:
                e = df
            else:
                r[f] = c0(v) - df
        o, p8 = p.narrow(dim + 1, 2, n), 1 / (8 * math.pi)
        et = o[0] * o[7] + 0.5 * o[0] * (o[1:4] ** 2).sum(0) + p8 * (o[4:7] ** 2).sum(0)
        r[7] = (et - e - 0.5 * r[0] * (r[1:4] ** 2).sum(0) - p8 * (r[4:7] ** 2).sum(0)) / r[0]
        return self.fill(out)

    def update(self, q, dt):
        ch2 = (0.8 * self.cfl * self.hmin / dt) ** 2
        argm = q
        for part in (4.0, 3.0, 2.0, 1.0):
            argm = self.stage(q, argm, dt / part, ch2, math.exp(-1 / (2 * part)))
        cc = sum(self.speeds(argm))
        for a in range(3):
            if self.n[a] > 1:
                argm = self.sweep(argm, cc, a, dt)
        return argm


def _exact_mhd(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    real = _np_dtype(case)
    kinds = ["periodic", "mirror" if case["bc"] == "mirror_y" else "periodic",
             "mirror" if case["bc"] == "mirror_z" else "periodic"]
    spacing = [real(real(b[1]) - real(b[0])) / real(k) for b, k in zip(_bounds(case), n)]
    sch = _Scheme(n, spacing, real, kinds)
    q = sch.fill(_initial(case, seed).double())
    dts = []
    for _ in range(case["steps"]):
        dts.append(sch.cfl_dt(q))
        q = sch.update(q, dts[-1])
    return {"q": q, "dt": dts}


# ------------------------------------------------------------------ ensemble
def _ensemble_sizes(case):
    return ensemble.kh_sizes(case["runs"], case["pick"])


def _ensemble_initial(n, seed, m):
    """Run m's (9, It, Jt, 1) state: a shear layer on [-0.5, 0.5]^2."""
    x = (torch.arange(n + 4, dtype=torch.float64, device=DEV) - 2 + 0.5) / n - 0.5
    rng = np.random.default_rng([seed, m])
    shape = (n + 4, n + 4, 1)
    q = torch.zeros((9,) + shape, dtype=torch.float64, device=DEV)
    t = torch.tanh(x / 0.02)[None, :, None].expand(shape)
    q[RO] = 1.5 - 0.5 * t
    q[VX] = 0.5 * t
    q[VY] = 1e-3 * (2 * torch.rand(shape, generator=_gen(1000003 * seed + m),
                                   dtype=torch.float64, device=DEV) - 1)
    q[BX] = rng.uniform(0.0, 0.2)
    q[EI] = 2.5 / 0.4 / q[RO]
    return q


def _prepare_ensemble(case, seed):
    ctx = mhd.ExecContext(0)
    sizes = _ensemble_sizes(case)
    ens = ensemble.Ensemble(ctx, [(n, n, 1) for n in sizes],
                            lambda m, g: _ensemble_initial(sizes[m], seed, m))
    ens.capture(case["steps"])
    return dict(ens=ens, steps=case["steps"])


def _run_ensemble(s):
    s["ens"].step(s["steps"])
    return [r.qq.data for r in s["ens"].runs]


def _exact_ensemble(case, seed):
    real, out = np.float32, []
    for m, n in enumerate(_ensemble_sizes(case)):
        d = real(real(0.5) - real(-0.5)) / real(n)
        sch = _Scheme((n, n, 1), (d, d, 1.0), real, ["periodic", "mirror", "periodic"], gm=1.4)
        q = sch.fill(_ensemble_initial(n, seed, m).float().double().permute(0, 3, 2, 1).contiguous())
        for _ in range(case["steps"]):
            q = sch.update(q, sch.cfl_dt(q))
        out.append(q)
    return out


# --------------------------------------------------------- radiative transfer
def _box_bounds(case):
    """The radiative box: unit height, cubic cells."""
    dz = 1.0 / case["nz"]
    return ((0.0, case["nx"] * dz), (0.0, case["ny"] * dz), (0.0, 1.0))


def _box_grid(case, device=DEV):
    return mhd.Grid(case["nx"], case["ny"], case["nz"], 2, bounds=_box_bounds(case),
                    dtype=np.float64, device=device)


def _strat():
    return rmhd.Stratification()


def _box_constants(case):
    z = (np.arange(case["nz"]) + 0.5) / case["nz"]
    s = _strat()
    kappa0 = s.kappa0(z, 1.0 / case["nz"])
    return s, kappa0, s.s_rad(z, kappa0)


def _box_state(case, seed, evolved=True):
    """The stratified box's (9, Kt, Jt, It) state; evolved: with the horizontal
    density and temperature structure that a few steps bring."""
    q = rmhd.stratified_box(_box_grid(case, "cpu"), _strat(), seed, device=DEV)
    q = q.permute(0, 3, 2, 1).contiguous()
    if evolved:
        rng = np.random.default_rng([seed, 3])
        x, y, z = ((torch.arange(case[k] + 4, dtype=torch.float64, device=DEV) - 1.5) / case[k]
                   for k in ("nx", "ny", "nz"))
        for f in (RO, EI):
            for _ in range(4):
                kx, ky, kz = rng.integers(1, 5, 3) * rng.choice([-1, 1], 3)
                wave = torch.sin(2 * math.pi * (kx * x[None, None, :] + ky * y[None, :, None]
                                                + kz * z[:, None, None]) + rng.uniform(0, 6.0))
                q[f] *= 1 + 0.01 * rng.normal() * wave
    return q


MU0 = 1 / 3
MU1 = math.sqrt(1 - 2 * MU0 * MU0)


def _exact_rt(q, n, dz, consts, faces, tolerance, max_iters):
    """Short characteristics along the 24 rays of the Carlson A4 set, every ray
    in its own mirrored frame in which it goes up all three axes.  Returns
    (iterations, intensities by ray (x, y, z), kappa, S, J - S on the lattice)."""
    s, kappa0, s_rad = consts
    lat = tuple(slice(1, 2 + k) for k in n)  # lattice nodes in x, y, z
    ro, ei = (q[f].permute(2, 1, 0)[lat] for f in (RO, EI))
    T = (s.gm - 1) * ei
    kap, src = (kappa0 * ro * T ** 3).contiguous(), (s_rad * T ** 4).contiguous()
    flips = [[a for a in range(3) if not (b >> a) & 1] for b in range(8)]
    k8 = torch.stack([kap.flip(f) for f in flips])
    s8 = torch.stack([src.flip(f) for f in flips])
    coef, axes = [], []
    for g in range(3):
        mu = [float(np.float32(MU1 if a == g else MU0)) for a in range(3)]
        ds = float(np.float32(min(dz / m for m in mu)))
        c = [m * ds / dz for m in mu]
        wb, wc = [c[a] for a in range(3) if a != g]
        w = ((1 - wb) * (1 - wc), wb * (1 - wc), (1 - wb) * wc, wb * wc)
        k, so = k8.movedim(g + 1, 1), s8.movedim(g + 1, 1)
        up = lambda f, w=w: (w[0] * f[..., 1:, 1:] + w[1] * f[..., :-1, 1:]  # noqa: E731
                             + w[2] * f[..., 1:, :-1] + w[3] * f[..., :-1, :-1])
        tau = 0.5 * (up(k[:, :-1]) + k[:, 1:, 1:, 1:]) * ds
        ex = torch.exp(-tau)
        u0 = 1 - ex
        u1 = torch.where(tau < 1e-4, 0.5 * tau, 1 - u0 / tau)
        coef.append((ex, (u0 - u1) * up(so[:, :-1]) + u1 * so[:, 1:, 1:, 1:]))
        axes.append(up)
    I = torch.zeros((3,) + tuple(k8.shape), dtype=torch.float64, device=DEV)
    it = 0
    while it < max_iters:
        old = I.clone()
        for a in (1, 0):  # x and y periodic: the far node enters again
            v = I.movedim(a + 2, 0)
            v[0] = v[-1].clone()
        for b in range(8):  # the z face the ray enters through
            kind = faces[0] if (b >> 2) & 1 else faces[1]
            I[:, b, :, :, 0] = s8[b, :, :, 0] if kind == 1 else 0.0
        for g in range(3):
            v = I[g].movedim(g + 1, 1)
            ex, em = coef[g]
            for p in range(1, v.shape[1]):
                v[:, p, 1:, 1:] = axes[g](v[:, p - 1]) * ex[:, p - 1] + em[:, p - 1]
        it += 1
        if float((I - old).abs().max().float()) < tolerance:
            break
    rays = torch.stack([I[g, b].flip(flips[b]) for g in range(3) for b in range(8)])
    return it, rays, kap, src, rays.sum(0) / 24 - src


def _on_lattice(f, n):
    """Lattice fields (.., x, y, z) in zero (.., Kt, Jt, It) fields."""
    out = torch.zeros(tuple(f.shape[:-3]) + tuple(k + 4 for k in reversed(n)),
                      dtype=torch.float64, device=DEV)
    out[..., 1:2 + n[2], 1:2 + n[1], 1:2 + n[0]] = f.transpose(-1, -3)
    return out


def _fields(grid, q):
    f = mhd.Fields(grid)
    f.data.copy_(q)
    return f


def _prepare_rt(case, seed):
    grid = _box_grid(case)
    return dict(ctx=mhd.ExecContext(0), rt=rt.RT(grid, 24), consts=_box_constants(case),
                qq=_fields(grid, _box_state(case, seed)))


def _run_rt(s):
    strat, kappa0, s_rad = s["consts"]
    r, ctx = s["rt"], s["ctx"]
    r.rint.zero_()
    r.source_from_fields(ctx, s["qq"], strat.gm, kappa0, s_rad)
    iters, _ = r.solve(ctx, tolerance=1e-6, max_iters=200, **rmhd.RT_FACES)
    q = r.qrad(ctx, tolerance=1e-6, max_iters=200, **rmhd.RT_FACES)
    return {"iters": iters, "qrad": q, "intensities": r.intensities()}


def _exact_rt_case(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    it, rays, kap, _, net = _exact_rt(_box_state(case, seed), n, 1.0 / case["nz"],
                                      _box_constants(case), (1, 2), 1e-6, 200)
    return {"iters": it, "qrad": _on_lattice(4 * math.pi * kap * net, n),
            "intensities": _on_lattice(rays, n)}


def _prepare_slab(case, seed):
    grid = _box_grid(case)
    q = _fields(grid, _box_state(case, seed))
    slab = rmhd.BottomSlabRT(grid, case["layers"], case["buffer"])
    return dict(ctx=mhd.ExecContext(0), slab=slab, consts=_box_constants(case), qq=q,
                q_full=torch.zeros_like(q.data[0]))


def _run_slab(s):
    strat, kappa0, s_rad = s["consts"]
    s["slab"].apply(s["ctx"], s["qq"], strat.gm, kappa0, s_rad, s["q_full"], tolerance=0.0,
                    max_iters=2)
    return {"qrad": s["q_full"], "rays": s["slab"].rt.intensities()}


def _exact_slab(case, seed):
    ls = case["layers"] + case["buffer"]
    n = (case["nx"], case["ny"], ls)
    q = _box_state(case, seed)[:, :ls + 4]
    _, rays, kap, _, net = _exact_rt(q, n, 1.0 / case["nz"], _box_constants(case), (1, 1), 0.0, 2)
    full = torch.zeros((case["nz"] + 4, case["ny"] + 4, case["nx"] + 4), dtype=torch.float64,
                       device=DEV)
    full[2:2 + case["layers"]] = _on_lattice(4 * math.pi * kap * net, n)[2:2 + case["layers"]]
    return {"qrad": full, "rays": _on_lattice(rays, n)}


# ------------------------------------------------------------- radiative MHD
def _prepare_rmhd(case, seed):
    box = rmhd.RadiativeMHD(_box_grid(case), mhd.ExecContext(0), _strat())
    box.initialize(seed)
    return dict(box=box)


def _run_rmhd(s):
    box = s["box"]
    dt = box.step_plain()
    return {"q": box.model.qq.data, "qrad": box.rt.qrad_field, "dt": dt}


def _exact_rmhd(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    s, kappa0, s_rad = consts = _box_constants(case)
    q0 = _box_state(case, seed, evolved=False)
    d = [np.float64(b[1]) / k for b, k in zip(_box_bounds(case), n)]
    sch = _Scheme(n, d, np.float64, ["periodic", "periodic", "fixed"], gm=s.gm, grav=s.grav,
                  fixed=q0.clone())
    q = sch.fill(q0.clone())
    _, rays, kap, _, net = _exact_rt(q, n, 1.0 / case["nz"], consts, (1, 2), 1e-6, 200)
    del rays
    qrad = _on_lattice(4 * math.pi * kap * net, n)
    dt = sch.cfl_dt(q)
    q = sch.update(q, dt)
    r = sch.inner(q)
    r[EI] += dt * sch.inner(qrad) / r[RO]
    return {"q": sch.fill(q), "qrad": qrad, "dt": dt}


# ----------------------------------------------------------------- surrogate
def _weights(nz, seed):
    rng = np.random.default_rng([seed, 5])
    sizes = [FEATURES * nz] + [HIDDEN] * HIDDEN_LAYERS + [nz]
    out = []
    for i, o in zip(sizes[:-1], sizes[1:]):
        out.append(((rng.standard_normal((o, i)) * math.sqrt(2 / i)).astype(np.float32),
                    (0.05 * rng.standard_normal(o)).astype(np.float32)))
    return out


def _surrogate(ctx, nz, seed, max_batch):
    sur = surrogate.ColumnSurrogate(ctx, nz, hidden=HIDDEN, hidden_layers=HIDDEN_LAYERS,
                                    max_batch=max_batch, device=DEV, features=FEATURES)
    for layer, (w, b) in enumerate(_weights(nz, seed)):
        hip.call("misohip_mlp_set_layer", ctx.handle, sur.h, layer,
                 w.ctypes.data_as(C.c_void_p), b.ctypes.data_as(C.c_void_p))
    return sur


def _raw_features(q, gm):
    """(columns, 4 nz) float64: ln ro, ln T, |B|^2 and the horizontal
    Laplacian of ln T of every interior column, x fastest over columns."""
    p = q[:, 2:-2, 2:-2, 2:-2].double()
    ln_t = torch.log((gm - 1) * p[EI])
    lap = -4 * ln_t
    for dim in (1, 2):
        for shift in (LAPLACIAN_STRIDE, -LAPLACIAN_STRIDE):
            lap = lap + ln_t.roll(shift, dim)
    f = torch.stack([torch.log(p[RO]), ln_t, (p[BX:BZ + 1] ** 2).sum(0), lap])
    return f.permute(2, 3, 0, 1).reshape(p.shape[2] * p.shape[3], -1)


def _norms(q, gm, nz):
    f = _raw_features(q, gm)
    mu, sd = f.mean(0), f.std(0).clamp_min(1e-6)
    z = np.arange(nz) / nz
    return [t.astype(np.float32) for t in (mu.cpu().numpy(), sd.cpu().numpy(),
                                           0.1 * np.sin(9 * z), 0.02 + 0.3 * np.exp(-8 * z))]


def _correction(case, seed):
    shape = tuple(case[k] + 4 for k in ("nz", "ny", "nx"))
    return 0.01 * torch.randn(shape, generator=_gen(seed + 77), dtype=torch.float64, device=DEV)


def _prepare_predict(case, seed):
    grid, ctx, gm = _box_grid(case), mhd.ExecContext(0), _strat().gm
    q = _fields(grid, _box_state(case, seed))
    sur = _surrogate(ctx, case["nz"], seed, case["nx"] * case["ny"] // 32 * 32 + 32)
    sur.set_normalization(*_norms(q.data, gm, case["nz"]))
    out = torch.zeros_like(q.data[0])
    return dict(sur=sur, grid=grid, qq=q, gm=gm, out=out, corr=_correction(case, seed))


def _run_predict(s):
    return s["sur"].predict(s["grid"], s["qq"], s["gm"], s["out"], corr=s["corr"])


def _bf(x):
    return x.to(torch.bfloat16).double()


def _silu(x):
    return x / (1 + torch.exp(-x))


def _exact_predict(case, seed):
    """The network as it is defined: bf16 weights and activations, everything
    between them in 64 bits."""
    gm, nz = _strat().gm, case["nz"]
    q = _box_state(case, seed)
    mu, sd, mu_o, sd_o = (torch.from_numpy(a).to(DEV).double() for a in _norms(q, gm, nz))
    x = _bf((_raw_features(q, gm) - mu) / sd)
    net = _weights(nz, seed)
    for layer, (w, b) in enumerate(net):
        x = x @ _bf(torch.from_numpy(w).to(DEV)).t() + torch.from_numpy(b).to(DEV).double()
        if layer < len(net) - 1:
            x = _bf(_silu(x))
    y = (x * sd_o + mu_o).reshape(case["ny"], case["nx"], nz).permute(2, 0, 1)
    out = torch.zeros_like(q[0])
    out[2:-2, 2:-2, 2:-2] = y + _correction(case, seed)[2:-2, 2:-2, 2:-2]
    return out


def _columns(case, seed):
    """Raw features and Q_rad columns: smooth height profiles with a few
    random amplitudes per column, Q_rad a smooth function of them."""
    g, nz, n = _gen(seed), case["nz"], case["columns"]
    z = torch.arange(nz, device=DEV, dtype=torch.float32) / nz
    basis = torch.stack([torch.cos(math.pi * k * z) / (1 + k) for k in range(12)])
    amp = torch.randn((n, FEATURES, 12), generator=g, device=DEV)
    feats = (amp @ basis).reshape(n, FEATURES * nz) * 0.1 - 1.0
    mix = torch.randn((FEATURES * 12, 12), generator=g, device=DEV) / 7
    targ = (torch.tanh(amp.reshape(n, -1) @ mix) @ basis) * torch.exp(-3 * z)
    return feats.contiguous(), targ.double().contiguous()


LR = 1e-3


def _prepare_fit(case, seed):
    ctx = mhd.ExecContext(0)
    feats, targ = _columns(case, seed)
    sur = _surrogate(ctx, case["nz"], seed, max(4096, case["batch"]))
    return dict(sur=sur, ctx=ctx, feats=feats, targ=targ, case=case)


def _run_fit(s):
    sur, c = s["sur"], s["case"]
    loss, val = sur.fit(s["feats"], s["targ"], epochs=c["epochs"], batch=c["batch"], lr=LR)
    out = {"val": val, "loss": loss}
    for layer, (i, o) in enumerate(zip(sur.sizes[:-1], sur.sizes[1:])):
        for which, shape in ((0, (o, i)), (1, (o,))):
            host = np.empty(shape, dtype=np.float32)
            hip.call("misohip_mlp_get_layer", s["ctx"].handle, sur.h, layer, which,
                     host.ctypes.data_as(C.c_void_p))
            out["%s%d" % ("wb"[which], layer)] = host
    return out


def _exact_fit(case, seed):
    feats, targ = _columns(case, seed)
    batch, epochs, n = case["batch"], case["epochs"], case["columns"]
    g = torch.Generator(device="cpu").manual_seed(0)
    perm = torch.randperm(n, generator=g).to(DEV)
    nval = max(batch, int(n * 0.1)) if n > 2 * batch else 0
    tr, va = perm[nval:], perm[:nval]
    ntr = (len(tr) // batch) * batch
    f64, t64 = feats[tr].double(), targ[tr].double()
    mu_i, mu_o, sd_o = f64.mean(0), t64.mean(0), t64.std(0).clamp_min(1e-12)
    sd_i = torch.maximum(f64.std(0), 1e-6 * f64.abs().mean(0)).clamp_min(1e-12)
    x_all, y_all = _bf((feats.double() - mu_i) / sd_i), (targ.double() - mu_o) / sd_o
    par = [[torch.from_numpy(t).to(DEV).double() for t in wb] for wb in _weights(case["nz"], seed)]
    mom = [[[torch.zeros_like(p), torch.zeros_like(p)] for p in wb] for wb in par]

    def forward(x):
        acts, pres = [x], []
        for layer, (w, b) in enumerate(par):
            pres.append(acts[-1] @ _bf(w).t() + b)
            acts.append(pres[-1] if layer == len(par) - 1 else _bf(_silu(pres[-1])))
        return acts, pres

    t, steps, loss = 0, epochs * (ntr // batch), 0.0
    for _ in range(epochs):
        order = tr[torch.randperm(len(tr), generator=g).to(DEV)][:ntr]
        for b0 in range(0, ntr, batch):
            sel = order[b0:b0 + batch]
            acts, pres = forward(x_all[sel])
            err = pres[-1] - y_all[sel]
            loss = float((err ** 2).mean())
            d = _bf(2 * err / err.numel())
            grads = []
            for layer in reversed(range(len(par))):
                grads.append((d.t() @ acts[layer], d.sum(0)))
                if layer:
                    sg = torch.sigmoid(pres[layer - 1])
                    d = _bf((d @ _bf(par[layer][0])) * sg * (1 + pres[layer - 1] * (1 - sg)))
            lr = 1e-5 + 0.5 * (LR - 1e-5) * (1 + math.cos(math.pi * t / max(1, steps)))
            t += 1
            for wb, ms, gs in zip(par, mom, reversed(grads)):
                for p, m, gr in zip(wb, ms, gs):
                    m[0] = 0.9 * m[0] + 0.1 * gr
                    m[1] = 0.999 * m[1] + 0.001 * gr * gr
                    p -= lr * (m[0] / (1 - 0.9 ** t)) / (torch.sqrt(m[1] / (1 - 0.999 ** t)) + 1e-8)
    out = {"loss": loss, "val": None}
    if nval:
        y = forward(x_all[va])[1][-1] * sd_o + mu_o
        out["val"] = float((y - targ[va]).norm() / targ[va].norm())
    for layer, (w, b) in enumerate(par):
        out["w%d" % layer], out["b%d" % layer] = w, b
    return out


# ----------------------------------------------------------------- interface
_FAMILIES = {
    "mhd": (_prepare_mhd, _run_mhd, _exact_mhd),
    "ensemble": (_prepare_ensemble, _run_ensemble, _exact_ensemble),
    "rmhd": (_prepare_rmhd, _run_rmhd, _exact_rmhd),
    "rt": (_prepare_rt, _run_rt, _exact_rt_case),
    "slab": (_prepare_slab, _run_slab, _exact_slab),
    "predict": (_prepare_predict, _run_predict, _exact_predict),
    "fit": (_prepare_fit, _run_fit, _exact_fit),
}


def prepare(case, seed):
    return case["kind"], _FAMILIES[case["kind"]][0](case, seed)


def run(state):
    kind, s = state
    return _FAMILIES[kind][1](s)


def exact(case, seed):
    return _FAMILIES[case["kind"]][2](case, seed)


def _step_work(cells, dims, size):
    """One MHD step: the state read once and written once (dt comes from a
    reduction over the whole state, so no two steps share a pass), and the
    arithmetic of four RK stages and `dims` viscosity sweeps."""
    return 18 * size * cells, cells * (4 * (200 * dims + 80) + 9 * 30 * dims)


# passes over the intensities that a solve takes: a cold one converges to the
# tolerance in about this many, a warm-started one in three
COLD_ITERS, WARM_ITERS = 8, 3


def _rt_work(nodes, iters):
    """`iters` sweeps of 24 rays: kappa and S read once a sweep, every
    intensity read (for the change) and written; then Q_rad."""
    return nodes * (iters * (24 * 16 + 16) + 24 * 8 + 24), nodes * 24 * (iters * 60 + 2)


def work(case):
    kind = case["kind"]
    if kind == "mhd":
        cells = case["nx"] * case["ny"] * case["nz"]
        b, f = _step_work(cells, 3 if case["nz"] > 1 else 2, 4 if case["dtype"] == "f32" else 8)
        return {"bytes": b * case["steps"], "flops": f * case["steps"]}
    if kind == "ensemble":
        b, f = _step_work(sum(n * n for n in _ensemble_sizes(case)), 2, 4)
        return {"bytes": b * case["steps"], "flops": f * case["steps"]}
    if kind == "fit":
        nz = case["nz"]
        weights = FEATURES * nz * HIDDEN + (HIDDEN_LAYERS - 1) * HIDDEN ** 2 + HIDDEN * nz
        cols = case["epochs"] * (int(case["columns"] * 0.9) // case["batch"]) * case["batch"]
        # the raw columns once; each step's batch and the weights' state
        return {"bytes": case["columns"] * nz * (4 * FEATURES + 8)
                + cols * nz * (2 * FEATURES + 4) + cols // case["batch"] * weights * 30,
                "flops": 6 * weights * cols}
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    cells = nx * ny * nz
    if kind == "predict":
        weights = FEATURES * nz * HIDDEN + (HIDDEN_LAYERS - 1) * HIDDEN ** 2 + HIDDEN * nz
        return {"bytes": 7 * 8 * cells, "flops": 2 * weights * nx * ny}
    if kind == "slab":
        nodes = (nx + 1) * (ny + 1) * (case["layers"] + case["buffer"] + 1)
        b, f = _rt_work(nodes, 2)
        return {"bytes": b + 8 * nx * ny * case["layers"], "flops": f}
    nodes = (nx + 1) * (ny + 1) * (nz + 1)
    b, f = _rt_work(nodes, COLD_ITERS if kind == "rt" else WARM_ITERS)
    if kind == "rt":
        return {"bytes": b + 24 * 16 * nodes, "flops": f}
    mb, mf = _step_work(cells, 3, 8)
    return {"bytes": b + mb, "flops": f + mf}
