"""The work this framework does for its users, as measurable cases.

Each case is one call pattern of the public entry points (``cubismup_3d_amd.Grid`` and
``cubismup_3d_amd.adjoint``) on a size its users run:

* ``loop``: a stretch of the device-resident step loop (``Grid.run_steps``) followed by the read-back of
  time, dt, max |u| and energy a driver logs, on periodic boxes: decaying or forced isotropic turbulence, the
  central and the upwind midpoint scheme, both precisions and both decompositions, a sphere in a stream.
* ``open``: the same call on boxes with open and wall faces (the sphere presets' dirichlet faces, a channel).
* ``freespace``: the operators one by one, as ``Simulation`` steps a box with freespace faces.
* ``adjoint``: the differentiable rollout and its backward.
* ``analysis``: the statistics written between stretches of steps (``Grid.diagnostics``, ``Grid.hit_analysis``).

``exact`` restates each case in 64 bits with plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import cubismup_3d_amd as cup
from cubismup_3d_amd.adjoint import kinetic_energy, rollout

BS = 8
TWO_PI = 2 * math.pi
PERIODIC = "periodic,periodic,periodic"
# cells per axis that every entry point takes: 8 x blocks, no prime factor above 5
LENGTHS = [n for n in range(16, 513, 8)
           if not [p for p in (7, 11, 13, 17, 19, 23, 29, 31, 37, 41, 43, 47, 53, 59, 61) if n % p == 0]]


def case(kind, nx, ny, nz, **kw):
    d = dict(kind=kind, nx=nx, ny=ny, nz=nz, precision=4, decomposition="fused", scheme=0, forced=False, steps=1,
             fixed_dt=0.0, nu=0.005, sphere=False, bc=PERIODIC)
    d.update(kw)
    return d


def listed():
    return [
        # the 64^3 Taylor-Green setting of the benchmark: fixed small steps, where launches count
        case("loop", 64, 64, 64, steps=20, fixed_dt=1e-3, nu=0.01, name="decay 64 f32"),
        # the headline: forced isotropic turbulence at 256^3, FP32
        case("loop", 256, 256, 256, forced=True, steps=10, name="forced 256 f32"),
        # the same with third-order upwind advection and the midpoint rule
        case("loop", 256, 256, 256, forced=True, scheme=2, steps=5, name="forced 256 f32 midpoint"),
        # a large DNS box: twice the headline's resolution
        case("loop", 512, 512, 512, forced=True, steps=2, nu=0.002, name="forced 512 f32"),
        # block counts that are no powers of two, as the DNS launch scripts' 12 blocks per side
        case("loop", 160, 96, 120, forced=True, steps=5, name="forced 160x96x120 f32"),
        # the fused loop in FP64, the accuracy runs' form
        case("loop", 128, 128, 128, precision=8, forced=True, steps=5, name="forced 128 f64"),
        # the reference's operator decomposition in FP64, the default of a double-precision Simulation
        case("loop", 128, 128, 128, precision=8, decomposition="plain", forced=True, steps=2,
             name="plain forced 128 f64"),
        # a penalized sphere held in a stream, Re = 200, at the drag gradient's grid
        case("loop", 256, 128, 128, steps=10, fixed_dt=1e-3, nu=1e-3, sphere=True, name="sphere 256x128x128 f32"),
        # the dissipated-energy gradient's rollout: forward and backward, two checkpoint segments
        case("adjoint", 128, 128, 128, steps=10, fixed_dt=2e-3, name="adjoint 128 f32"),
        # a box with the sphere presets' dirichlet faces and a wall pair
        case("open", 128, 96, 64, precision=8, decomposition="plain", steps=2, nu=0.01,
             bc="dirichlet,wall,periodic", name="open 128x96x64 f64"),
        # freespace faces: the unbounded pressure solve, operator by operator
        case("freespace", 64, 64, 64, precision=8, decomposition="plain", steps=2, nu=0.01,
             bc="freespace,freespace,freespace", name="freespace 64 f64"),
        # the analysis written between stretches of steps
        case("analysis", 128, 128, 128, name="analysis 128 f32"),
    ]


def _length(rng, lo, hi):
    want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min((n for n in LENGTHS if lo <= n <= hi), key=lambda n: abs(math.log(n / want)))


def draw(rng):
    kind = rng.choice(["loop", "loop", "loop", "sphere", "adjoint", "open", "freespace", "analysis"])
    top = {"loop": 400, "sphere": 256, "adjoint": 160, "open": 192, "freespace": 128, "analysis": 256}[kind]
    n = _length(rng, 64 if kind == "sphere" else 32, top)
    if rng.random() < 0.4:
        dims = [n, n, n]
    else:
        dims = [n] + [_length(rng, max(16, n // 2), n) for _ in range(2)]
        if kind != "sphere":
            rng.shuffle(dims)
    precision = rng.choice([4, 4, 8])
    steps = rng.choice([1, 2, 3, 5, 8])
    if kind == "sphere":
        dims[1:] = [max(d, 48) for d in dims[1:]]
        return case("loop", *dims, precision=precision, steps=steps, fixed_dt=1e-3, nu=1e-3, sphere=True,
                    decomposition=rng.choice(["fused", "fused", "plain"]))
    if kind == "adjoint":
        return case("adjoint", *dims, precision=precision, steps=rng.choice([2, 4, 6, 10]), fixed_dt=2e-3,
                    scheme=rng.choice([0, 0, 2]))
    if kind == "open":
        bc = rng.choice(["dirichlet,dirichlet,dirichlet", "dirichlet,wall,periodic", "periodic,wall,periodic",
                         "wall,wall,wall", "periodic,dirichlet,wall"])
        return case("open", *dims, precision=precision, decomposition="plain", steps=min(steps, 3), nu=0.01, bc=bc)
    if kind == "freespace":
        return case("freespace", *dims, precision=precision, decomposition="plain", steps=min(steps, 3), nu=0.01,
                    bc="freespace,freespace,freespace")
    if kind == "analysis":
        return case("analysis", *dims, precision=precision)
    forced = rng.random() < 0.6
    scheme, decomposition = rng.choice([0, 0, 2]), rng.choice(["fused", "fused", "plain"])
    weight = precision / 4 * (2 if scheme else 1) * (6 if decomposition == "plain" else 1)
    most = int(2 * 512 ** 3 / (dims[0] * dims[1] * dims[2] * weight))
    return case("loop", *dims, precision=precision, forced=forced, steps=max(1, min(steps, most)), scheme=scheme,
                decomposition=decomposition, fixed_dt=0.0 if forced else 1e-3)


# ---------------------------------------------------------------------------- inputs


def _extent(c):
    """The box's longest side: 2 pi, or 2 with the sphere and 1 with non-periodic faces."""
    return 2.0 if c["sphere"] else (TWO_PI if c["bc"] == PERIODIC else 1.0)


def _uinf(c):
    return (1.0, 0.0, 0.0) if c["sphere"] else ((0.3, -0.2, 0.1) if c["bc"] != PERIODIC else (0.0, 0.0, 0.0))


SPHERE_D, SPHERE_LAMBDA, CFL = 0.2, 1e6, 0.3


def _sphere_center(c):
    h = _extent(c) / max(c["nx"], c["ny"], c["nz"])
    return (0.5, 0.5 * c["ny"] * h, 0.5 * c["nz"] * h)


def _dtype(c):
    return torch.float32 if c["precision"] == 4 else torch.float64


def _velocity(c, seed):
    """Solenoidal random-phase velocity [3][Z][Y][X] with E(k) ~ k^4 exp(-2 (k/k0)^2), k0 = 4 wavelengths in
    the longest side, scaled to u_rms = 1 (0.1 about the sphere's stream)."""
    shape = (c["nz"], c["ny"], c["nx"])
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    k = [torch.fft.fftfreq(n, 1.0 / n, device="cuda") for n in shape[:2]]
    k.append(torch.fft.rfftfreq(shape[2], 1.0 / shape[2], device="cuda"))
    longest = max(shape)
    kz, ky, kx = [(longest / n * q).to(_dtype(c)) for n, q in zip(shape, k)]
    kk = (kz[:, None, None], ky[None, :, None], kx[None, None, :])
    k2 = kk[0] ** 2 + kk[1] ** 2 + kk[2] ** 2
    amp = k2.sqrt() * torch.exp(-k2 / 16.0)
    hat = [torch.fft.rfftn(torch.randn(shape, generator=gen, device="cuda", dtype=_dtype(c))) * amp for _ in range(3)]
    dot = (kk[2] * hat[0] + kk[1] * hat[1] + kk[0] * hat[2]) / k2.clamp_min(1e-30)
    u = torch.stack([torch.fft.irfftn(hat[q] - kk[2 - q] * dot, s=shape) for q in range(3)])
    del hat, dot
    rms = 0.1 if c["sphere"] else 1.0
    return u * (rms / (u * u).mean().sqrt())


def _target(u):
    """The velocity's kinetic energy per volume, which the forcing holds."""
    return 0.5 * sum(float((q * q).mean(dtype=torch.float64)) for q in u)


class _Field:
    """A field's device buffer for torch (zero copy); holds the grid, which owns the buffer."""

    def __init__(self, g, name):
        self.grid = g
        self.__cuda_array_interface__ = dict(shape=(g.bpd[2], g.bpd[1], g.bpd[0], BS, BS, BS), version=2, strides=None,
                                             typestr="<f%d" % g.precision, data=(g.device_ptr(name), False))


def _views(g):
    """u, v, w, p as the grid holds them: [block z][block y][block x][8][8][8]. The buffers are the grid's, so
    each tensor keeps it alive: a caller may hold a pass's outputs longer than the state."""
    out = {n: torch.as_tensor(_Field(g, n), device="cuda") for n in "uvwp"}
    for t in out.values():
        t.grid = g
    return out


def prepare(c, seed):
    u = _velocity(c, seed)
    g = cup.Grid((c["nx"] // BS, c["ny"] // BS, c["nz"] // BS), maxextent=_extent(c), precision=c["precision"],
                 decomposition=c["decomposition"], bc=tuple(c["bc"].split(",")))
    s = dict(c=c, g=g, uinf=_uinf(c))
    if c["sphere"]:
        g.chi_from_sphere(_sphere_center(c), SPHERE_D / 2)
        s["sphere"] = dict(lambda_=SPHERE_LAMBDA, implicit=True, trans_vel=(-1.0, 0.0, 0.0))
    if c["kind"] == "adjoint":
        s["u0"] = u.requires_grad_(True)
        return s
    g.set_torch_velocity(u)
    s["target"] = _target(u) if c["forced"] else 0.0
    if c["kind"] == "analysis":  # a state of the run: one step sets the pressure
        g.run_steps(1, nu=c["nu"], fixed_dt=1e-3)
    s["views"] = _views(g)
    return s


# ---------------------------------------------------------------------------- one pass


def run(s):
    return {"loop": _run_loop, "open": _run_loop, "freespace": _run_operators, "adjoint": _run_adjoint,
            "analysis": _run_analysis}[s["c"]["kind"]](s)


def _numbers(c, values):
    return np.asarray(values, dtype=np.float32 if c["precision"] == 4 else np.float64)


def _run_loop(s):
    c, g = s["c"], s["g"]
    g.run_steps(c["steps"], CFL=CFL, nu=c["nu"], uinf=s["uinf"], fixed_dt=c["fixed_dt"], scheme=c["scheme"],
                spectral_forcing=c["forced"], tke_target=s["target"], sphere=s.get("sphere"))
    st = g.step_state()
    out = dict(s["views"], time=_numbers(c, st["time"]), dt=_numbers(c, st["last_dt"]))
    if c["decomposition"] == "fused":
        out.update(umax=_numbers(c, st["umax"]), ke=_numbers(c, st["ke"]))
    if c["sphere"]:
        out["force"] = _numbers(c, g.last_body_force())
    return out


def _run_operators(s):
    c, g = s["c"], s["g"]
    for _ in range(c["steps"]):
        dt, umax = g.calc_max_timestep(CFL, c["nu"], s["uinf"])
        g.advect_diffuse(dt, c["nu"], s["uinf"])
        g.pressure_rhs(dt)
        g.poisson_unbounded()
        g.pressure_project(dt)
    return dict(s["views"], dt=_numbers(c, dt), umax=_numbers(c, umax))


def _run_adjoint(s):
    c, g, u0 = s["c"], s["g"], s["u0"]
    un = rollout(u0, g, c["steps"], c["nu"], dts=[c["fixed_dt"]] * c["steps"], every=max(1, c["steps"] // 2),
                 scheme=c["scheme"])
    (grad,) = torch.autograd.grad(kinetic_energy(un, g.h), u0)
    return un.detach(), grad


def _run_analysis(s):
    c, g = s["c"], s["g"]
    a = g.hit_analysis(c["nu"])
    return dict(diagnostics=_numbers(c, g.diagnostics(c["nu"])), spectrum=_numbers(c, a["E"]),
                stats=_numbers(c, [a[k] for k in ("tke", "eps", "uprime", "lambda", "Re_lambda", "l_integral",
                                                  "tau_integral", "grad_mean", "grad_std")]))


# ---------------------------------------------------------------------------- what a pass cannot do without


def work(c):
    """Bytes: the velocity read and written and the pressure written once a step (a step couples every cell with
    every other, so the next one reads them again); the adjoint's backward reads the state and the adjoint and
    writes the adjoint. Operations: the stencils' and one forward and one inverse transform's."""
    n = c["nx"] * c["ny"] * c["nz"]
    e = c["precision"]
    fft = 2.5 * n * math.log2(n)
    if c["kind"] == "analysis":
        return dict(bytes=4 * n * e, flops=3 * fft + 150 * n)
    step_flops = (120 if c["scheme"] == 0 else 320) * n + 2 * fft * (8 if c["kind"] == "freespace" else 1)
    if c["kind"] == "adjoint":
        return dict(bytes=c["steps"] * (7 + 10) * n * e, flops=c["steps"] * 3 * step_flops)
    return dict(bytes=c["steps"] * 7 * n * e, flops=c["steps"] * step_flops)


# ---------------------------------------------------------------------------- the same in 64 bits


class _Box:
    """The step's operators in plain torch, FP64, on arrays [Z][Y][X] (axis d of x, y, z is dimension 2 - d)."""

    def __init__(self, c):
        self.c = c
        self.n = (c["nx"], c["ny"], c["nz"])
        self.bc = c["bc"].split(",")
        self.h = _extent(c) / max(self.n)
        self.uinf = _uinf(c)

    def shift(self, f, d, k, sign=1.0, fade=None):
        """f at the cell k along axis d, through the faces: the periodic image, or the boundary cell (negated at
        a wall with sign = -1, times the face's fade where one is given)."""
        dim = 2 - d
        g = torch.roll(f, -k, dim)
        if self.bc[d] == "periodic":
            return g
        edge = f.select(dim, f.shape[dim] - 1 if k > 0 else 0)
        s = sign if self.bc[d] == "wall" else (1.0 if fade is None else fade[2 * d + (k > 0)])
        g.select(dim, f.shape[dim] - 1 if k > 0 else 0).copy_(edge * s)
        return g

    def fades(self, umax, dt):
        fac = min(1.0, umax * dt / self.h)
        nor = max([abs(x) for x in self.uinf] + [2.0 ** -52])
        return [1 - fac * (f(x, 0.0) / nor) ** 2 for x in self.uinf for f in (max, min)]

    def max_u(self, u):
        return max(float((u[q] + self.uinf[q]).abs().max()) for q in range(3))

    def cfl(self, umax):
        return CFL * min(self.h * self.h / self.c["nu"], self.h / (umax + 1e-8))

    def central(self, u, dt, fade=None):
        out = []
        for q in range(3):
            adv, lap = 0, -6 * u[q]
            for d in range(3):
                p, m = (self.shift(u[q], d, k, -1.0, fade) for k in (1, -1))
                adv = adv + (u[d] + self.uinf[d]) * (p - m)
                lap = lap + p + m
            out.append(u[q] - dt / (2 * self.h) * adv + self.c["nu"] * dt / self.h ** 2 * lap)
        return torch.stack(out)

    def upwind(self, s, base, dt):
        out = []
        for q in range(3):
            adv, lap, f = 0, -6 * s[q], s[q]
            for d in range(3):
                m2, m1, p1, p2 = (self.shift(f, d, k) for k in (-2, -1, 1, 2))
                a = s[d] + self.uinf[d]
                adv = adv + a * torch.where(a > 0, 2 * p1 + 3 * f - 6 * m1 + m2, -p2 + 6 * p1 - 3 * f - 2 * m1)
                lap = lap + m1 + p1
            out.append(base[q] - dt / (6 * self.h) * adv + self.c["nu"] * dt / self.h ** 2 * lap)
        return torch.stack(out)

    def advect(self, u, dt, umax=0.0):
        if self.c["scheme"] == 2:
            return self.upwind(self.upwind(u, u, dt / 2), u, dt)
        if self.c["bc"] == PERIODIC:
            return self.central(u, dt)
        u = self.central(u, dt, self.fades(umax, dt))
        opened = [d for d in range(3) if self.bc[d] in ("dirichlet", "freespace")]
        flux = sum(float(u[d].select(2 - d, -1).sum() - u[d].select(2 - d, 0).sum()) for d in opened)
        nx, ny, nz = self.n
        corr = flux / (2 * (nx * ny + nx * nz + ny * nz))
        if opened and abs(corr) >= 2.0 ** -52:
            for d in opened:
                u[d].select(2 - d, 0).add_(corr)
                u[d].select(2 - d, -1).sub_(corr)
        return u

    def force(self, u, target):
        shape = u.shape[1:]
        freq = [(torch.fft.fftfreq if i < 2 else torch.fft.rfftfreq)(m, 1.0 / m, device=u.device, dtype=torch.float64)
                * (TWO_PI / (m * self.h)) for i, m in enumerate(shape)]
        k2 = freq[0][:, None, None] ** 2 + freq[1][None, :, None] ** 2 + freq[2][None, None, :] ** 2
        band = (k2 > 0) & (k2 <= 4)
        low = torch.stack([torch.fft.irfftn(torch.fft.rfftn(u[q]) * band, s=shape) for q in range(3)])
        n = u[0].numel()
        tke, tke_low = (float((f * f).sum()) / (2 * n) for f in (u, low))
        fac = (target - tke) / (2 * tke_low)
        return u + fac * low if fac > 0 else u

    def rhs(self, u, dt):
        div = sum(self.shift(u[d], d, 1, -1.0) - self.shift(u[d], d, -1, -1.0) for d in range(3))
        return 0.5 * self.h * self.h / dt * div

    def poisson(self, r):
        if self.c["kind"] == "freespace":
            return self.poisson_free(r)
        if self.c["bc"] != PERIODIC:
            return self.poisson_mixed(r)
        freq = [torch.arange(m // 2 + 1 if i == 2 else m, device=r.device, dtype=torch.float64) / m
                for i, m in enumerate(r.shape)]
        cz, cy, cx = (torch.cos(4 * math.pi * f) for f in freq)
        den = 2 * (cz[:, None, None] + cy[None, :, None] + cx[None, None, :]) - 6
        ends = [torch.zeros(f.numel(), dtype=torch.bool, device=r.device) for f in freq]
        for e, m in zip(ends, r.shape):
            e[0] = e[m // 2] = True
        zero = ends[0][:, None, None] & ends[1][None, :, None] & ends[2][None, None, :]
        sym = torch.where(zero, torch.zeros_like(den), 4 / (self.h * torch.where(zero, torch.ones_like(den), den)))
        return torch.fft.irfftn(torch.fft.rfftn(r) * sym, s=r.shape)

    def poisson_mixed(self, r):
        tol, den, back, norm = 0.01, [], [], 1 / self.h
        for d, n in enumerate(self.n):
            dim = 2 - d
            per = self.bc[d] == "periodic"
            i = torch.arange(n, device=r.device, dtype=torch.float64)
            j, k = i[:, None], i[None, :]
            if per:  # the half-complex transform of the real line: cosines up to n/2, then sines
                low = k <= n // 2
                fw = torch.where(low, torch.cos(TWO_PI * j * k / n), -torch.sin(TWO_PI * j * (n - k) / n))
                bw = torch.where(j <= n // 2, torch.cos(TWO_PI * j * k / n), -torch.sin(TWO_PI * (n - j) * k / n))
                bw = bw * torch.where((j == 0) | (2 * j == n), 1.0, 2.0)
                kk, half, wf = torch.where(i <= n // 2, i, n - i), 0.0, TWO_PI / n
            else:    # DCT-II and DCT-III
                fw = 2 * torch.cos(math.pi * (j + 0.5) * k / n)
                bw = torch.cos(math.pi * j * (k + 0.5) / n) * torch.where(j == 0, 1.0, 2.0)
                kk, half, wf = i, 0.5, math.pi / n
            r = torch.movedim(torch.movedim(r, dim, 2).contiguous().reshape(-1, n).mm(fw).reshape(
                [m for q, m in enumerate(r.shape) if q != dim] + [n]), 2, dim)
            back.append((dim, n, bw))
            den.append((1 - tol) * (torch.cos(2 * wf * i) - 1) / 2 - tol * ((kk + half) * wf) ** 2)
            norm *= (1.0 if per else 0.5) / n
        total = den[2][:, None, None] + den[1][None, :, None] + den[0][None, None, :]
        r = r * (norm / total)
        r[0, 0, 0] = 0
        for dim, n, bw in back:
            r = torch.movedim(torch.movedim(r, dim, 2).contiguous().reshape(-1, n).mm(bw).reshape(
                [m for q, m in enumerate(r.shape) if q != dim] + [n]), 2, dim)
        return r.contiguous()

    def poisson_free(self, r):
        size = [2 * m for m in r.shape]
        dist = [torch.minimum(i, m - i) for m, i in
                ((m, torch.arange(m, device=r.device, dtype=torch.float64)) for m in size)]
        rr = (dist[0][:, None, None] ** 2 + dist[1][None, :, None] ** 2 + dist[2][None, None, :] ** 2).sqrt()
        green = torch.where(rr > 0, -1 / (4 * math.pi * self.h * rr.clamp_min(1e-30)), -0.1924173658 / self.h)
        p = torch.fft.irfftn(torch.fft.rfftn(r, s=size) * torch.fft.rfftn(green), s=size)
        return p[:r.shape[0], :r.shape[1], :r.shape[2]].contiguous()

    def project(self, u, p, dt):
        return torch.stack([u[d] - dt / (2 * self.h) * (self.shift(p, d, 1) - self.shift(p, d, -1))
                            for d in range(3)])


class _Ball:
    """The sphere's smoothed chi, the masking of the pressure RHS and the penalization, FP64."""

    def __init__(self, box):
        c, h = box.c, box.h
        self.box = box
        x, y, z = ((torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) * h for n in box.n)
        self.x = torch.broadcast_tensors(x[None, None, :], y[None, :, None], z[:, None, None])
        ctr = _sphere_center(c)
        sdf = SPHERE_D / 2 - sum((a - b) ** 2 for a, b in zip(self.x, ctr)).sqrt()
        g_u, g_i = [], []
        for d in range(3):
            p, m = torch.roll(sdf, -1, 2 - d), torch.roll(sdf, 1, 2 - d)
            g_u.append((p - m) / (2 * h))
            g_i.append((p.clamp_min(0) - m.clamp_min(0)) / (2 * h))
        smooth = sum(a * b for a, b in zip(g_i, g_u)) / (sum(a * a for a in g_u) + 2.0 ** -52)
        self.chi = torch.where(sdf.abs() > 2 * h, (sdf > 0).double(), smooth)
        stored = self.chi.to(_dtype(c)).double()
        grad = [torch.roll(stored, -1, 2 - d) - torch.roll(stored, 1, 2 - d) for d in range(3)]
        self.surface = sum(a * a for a in grad) > 0
        mass = self.chi.sum()
        self.arm = [a - (self.chi * a).sum() / mass for a in self.x]

    def mask(self, r):
        bulk = -self.chi * r
        r = r + bulk
        total, on = float(bulk.sum()), r[self.surface]
        part = float(on[on > 0].sum() if total > 0 else -on[on < 0].sum())
        corr = total / max(part, 2.0 ** -52)
        hit = self.surface & ((r > 0) if corr > 0 else (r < 0) if corr < 0 else torch.zeros_like(self.surface))
        return torch.where(hit, r - abs(corr) * r, r)

    def penalize(self, u, dt):
        pf = self.chi * SPHERE_LAMBDA / (1 + SPHERE_LAMBDA * dt * self.chi)
        f = [pf * (v - u[d]) for d, v in enumerate((-1.0, 0.0, 0.0))]
        dv, (x, y, z) = self.box.h ** 3, self.arm
        out = [f[0], f[1], f[2], y * f[2] - z * f[1], z * f[0] - x * f[2], x * f[1] - y * f[0]]
        return u + dt * torch.stack(f), [dv * float(q.sum()) for q in out]


def _blocks(f):
    z, y, x = f.shape
    return f.reshape(z // BS, BS, y // BS, BS, x // BS, BS).permute(0, 2, 4, 1, 3, 5).contiguous()


def exact(c, seed):
    """What run() returns for these inputs, in 64 bits with plain torch."""
    box = _Box(c)
    u = _velocity(c, seed).double()
    if c["kind"] == "adjoint":
        return _exact_adjoint(box, u)
    if c["kind"] == "analysis":
        return _exact_analysis(box, u)
    target = _target(u)
    ball = _Ball(box) if c["sphere"] else None
    time, force, p = 0.0, None, None
    for _ in range(c["steps"]):
        umax = box.max_u(u)
        dt = c["fixed_dt"] if c["fixed_dt"] > 0 else box.cfl(umax)
        u = box.advect(u, dt, 0.0 if c["fixed_dt"] > 0 else umax)
        if c["forced"]:
            u = box.force(u, target)
        r = box.rhs(u, dt)
        p = box.poisson(ball.mask(r) if ball else r)
        u = box.project(u, p, dt)
        if ball:
            u, force = ball.penalize(u, dt)
        time += dt
    out = dict(zip("uvwp", (_blocks(f) for f in (u[0], u[1], u[2], p))), dt=np.float64(dt))
    if c["kind"] == "freespace":
        return dict(out, umax=np.float64(umax))
    out["time"] = np.float64(time)
    if c["decomposition"] == "fused":
        out.update(umax=np.float64(box.max_u(u)), ke=np.float64(0.5 * box.h ** 3 * float((u * u).sum())))
    if c["sphere"]:
        out["force"] = np.asarray(force)
    return out


def _exact_adjoint(box, u0):
    """Reverse steps with the gradient of each by torch's autograd from the stored states."""
    c, dt = box.c, box.c["fixed_dt"]

    def step(u):
        u = box.advect(u, dt)
        return box.project(u, box.poisson(box.rhs(u, dt)), dt)

    states = [u0]
    with torch.no_grad():
        for _ in range(c["steps"]):
            states.append(step(states[-1]))
    lam = box.h ** 3 * states[-1]
    for s in reversed(states[:-1]):
        s = s.detach().requires_grad_(True)
        (lam,) = torch.autograd.grad(step(s), s, lam)
    return states[-1], lam


def _exact_analysis(box, u):
    c, h, nu = box.c, box.h, box.c["nu"]
    dt = 1e-3
    u = box.advect(u, dt)
    p = box.poisson(box.rhs(u, dt))
    u = box.project(u, p, dt)

    def der(f, d):
        return (torch.roll(f, -1, 2 - d) - torch.roll(f, 1, 2 - d)) / (2 * h)

    def lap(f):
        return sum(torch.roll(f, -1, d) + torch.roll(f, 1, d) for d in range(3)).sub(6 * f) / (h * h)

    dv = h ** 3
    x, y, z = ((torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) * h - 0.5 * n * h for n in box.n)
    x, y, z = torch.broadcast_tensors(x[None, None, :], y[None, :, None], z[:, None, None])
    D = [[der(u[q], d) for d in range(3)] for q in range(3)]
    w = [D[2][1] - D[1][2], D[0][2] - D[2][0], D[1][0] - D[0][1]]
    strain = sum(((D[i][j] + D[j][i]) / 2) ** 2 for i in range(3) for j in range(3))
    visc = sum(lap(u[q]) * u[q] for q in range(3)) + 2 * strain
    power = -sum(der(p, d) * u[d] for d in range(3))
    terms = [w[0], w[1], w[2], (y * w[2] - z * w[1]) / 2, (z * w[0] - x * w[2]) / 2, (x * w[1] - y * w[0]) / 2,
             u[0], u[1], u[2], (x * (y * w[1] + z * w[2]) - w[0] * (y * y + z * z)) / 3,
             (y * (x * w[0] + z * w[2]) - w[1] * (x * x + z * z)) / 3,
             (z * (x * w[0] + y * w[1]) - w[2] * (x * x + y * y)) / 3,
             y * u[2] - z * u[1], z * u[0] - x * u[2], x * u[1] - y * u[0], power, nu * visc,
             sum(a * b for a, b in zip(w, u)), (u * u).sum(0) / 2, sum(a * a for a in w).sqrt()]
    diag = [dv * float(t.sum()) for t in terms[:-1]] + [float(terms[-1].sum())]
    grad2 = sum(D[q][d] ** 2 for q in range(3) for d in range(3))
    gmean, gsq = float(grad2.sqrt().mean()), float(grad2.mean())
    # the shell spectrum and the spectral statistics
    shape, n = u.shape[1:], u[0].numel()
    idx = [(torch.fft.fftfreq if i < 2 else torch.fft.rfftfreq)(m, 1.0 / m, device=u.device, dtype=torch.float64)
           for i, m in enumerate(shape)]
    iz, iy, ix = idx[0].abs()[:, None, None], idx[1].abs()[None, :, None], idx[2].abs()[None, None, :]
    wx = torch.full((shape[2] // 2 + 1,), 2.0, device=u.device, dtype=torch.float64)
    wx[0] = wx[-1] = 1
    e = 0.5 * wx * sum(torch.fft.rfftn(u[q]).abs() ** 2 for q in range(3)) / n ** 2
    tke = float(e.sum())
    k = sum((TWO_PI / (m * h) * i) ** 2 for m, i in zip(shape, (iz, iy, ix))).sqrt()
    lint = float(torch.where(k > 0, e / k.clamp_min(1e-30), 0.0).sum()) / tke
    eps = nu * float(sum(a * a for a in w).mean())
    k2 = iz ** 2 + iy ** 2 + ix ** 2
    nyq = max(shape) // 2
    shell = torch.floor(k2.sqrt() * ((nyq - 1) / nyq)).long()
    live = k2 < nyq * nyq
    spectrum = torch.bincount(shell.expand_as(e)[live.expand_as(e)], weights=e[live.expand_as(e)],
                              minlength=nyq - 1)[:nyq - 1]
    up = math.sqrt(2 * tke / 3)
    taylor = math.sqrt(15 * nu / eps) * up
    return dict(diagnostics=np.asarray(diag), spectrum=spectrum.cpu().numpy(),
                stats=np.asarray([tke, eps, up, taylor, up * taylor / nu, lint, lint / up, gmean,
                                  math.sqrt(gsq - gmean ** 2)]))
