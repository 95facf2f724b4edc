"""The work that a user of this framework has it do, as measurable cases.

One case is a dict of plain values; `prepare` makes what a program has in
hand (plan, solver, state on the GPU), `run` is one pass through the public
entry points, `exact` is the same pass in plain torch FP64.  The families:

  dns      a DNS solver stepped `steps` steps (IF-RK4 or IF-AB2; unforced,
           constant-power or helical forcing; static or dynamic Smagorinsky;
           passive scalar; FP32 or FP64); the state on the device comes back
  ens2d    a batch of 2D ensemble members stepped and read back to the host
           (IF-RK4 vorticity scheme, or the phase-shift dealiased one)
  adjoint  forward map and gradient through torch.autograd
  rhs      the RHS of the reference's routine interface on host arrays
"""
import math

import numpy as np
import torch

import speccodelib_amd as scl
from speccodelib_amd import torch_adjoint

DEV = "cuda"


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------
def dns(nx, ny, nz, **kw):
    c = dict(kind="dns", nx=nx, ny=ny, nz=nz, prec="sp", steps=10, stepper=0, forced=1, sgs=0, scalar=False,
             nu=0.01, dt=0.002, kcut=0.0)
    c.update(kw)
    return c


def ens(scheme, groups, **kw):
    c = dict(kind="ens2d", scheme=scheme, groups=" ".join(f"{n}x{m}" for n, m in groups), steps=100)
    c.update(kw)
    return c


def listed():
    return [
        # smallest call: a 32^3 test-size DNS advanced one step at a time
        # (a driver that looks at the flow every step); launches dominate
        dict(dns(32, 32, 32, steps=1), name="dns_32_one_step"),
        # an ordinary production-size run between two outputs
        dict(dns(128, 128, 128), name="dns_128"),
        # the headline configuration: 512^3 forced DNS
        dict(dns(512, 512, 512, steps=5), name="dns_512"),
        # double precision on an uneven box, decaying turbulence
        dict(dns(64, 256, 128, prec="dp", forced=0), name="dns_box_fp64"),
        # helical forcing on a long box: the 1024-point lines of the largest
        # DNS configuration on a grid of 33M points
        dict(dns(256, 128, 1024, forced=2, nu=5e-4, dt=1e-3, steps=5), name="heli_box_1024"),
        # the production drivers' stepper: CFL steps, truncation at nx/2 - 1
        dict(dns(256, 256, 256, stepper=1, kcut=127.0, steps=20), name="ab2_256"),
        # static Smagorinsky LES with a passive scalar, the 256^3 configuration
        dict(dns(256, 256, 256, sgs=1, scalar=True, nu=1e-4, dt=1e-3, steps=5), name="les_scalar_256"),
        # dynamic Smagorinsky LES (coefficient every 10 steps)
        dict(dns(64, 64, 64, sgs=2, nu=5e-3, dt=2e-3, steps=20), name="les_dynamic_64"),
        # the three-size 2D ensemble batch, stepped and read back
        dict(ens(0, [(256, 192), (512, 48), (1024, 16)]), name="ens2d_batch"),
        # a few members of the phase-shift scheme, odd counts
        dict(ens(1, [(128, 7), (512, 3)], steps=200), name="turb2d_small"),
        # gradient of a 20-step LES map (data assimilation): forward + backward
        dict(kind="adjoint", nx=64, ny=64, nz=64, sgs=1, steps=20, ckpt=10, nu=5e-3, dt=2e-3, name="adjoint_les_64"),
        # the reference's RHS routine called on host arrays (drop-in linking)
        dict(kind="rhs", nx=128, ny=128, nz=128, prec="sp", forced=1, name="rhs_host_128"),
    ]


def draw(rng):
    """One more case of the ranges above: every family, grid axes 16..1024
    (spread over their logarithm), up to the largest listed case's work."""
    def log_pow2(lo, hi):
        return 1 << rng.randint(lo, hi)

    kind = rng.choice(["dns", "dns", "dns", "ab2", "les", "ens2d", "turb2d", "adjoint", "rhs"])
    eps = rng.uniform(0.7, 1.4)
    if kind in ("dns", "ab2", "les", "rhs"):
        prec = rng.choice(["sp", "sp", "sp", "dp"])
        top = {"dns": 26, "ab2": 26, "les": 24, "rhs": 22}[kind] - (2 if prec == "dp" else 0)
        while True:
            n = [log_pow2(4, 10) for _ in range(3)]
            if 14 <= sum(a.bit_length() - 1 for a in n) <= top:
                break
        if kind == "rhs":
            return dict(kind="rhs", nx=n[0], ny=n[1], nz=n[2], prec=prec, forced=rng.choice([0, 1, 2]), eps=0.1 * eps)
        big = max(n)
        kw = dict(prec=prec, steps=rng.randint(1, 10), forced=rng.choice([0, 1, 1, 2]), nu=0.5 * eps / big,
                  dt=0.25 * eps / big)
        if kind == "ab2":
            kw.update(stepper=rng.choice([1, 1, 2]), kcut=rng.choice([0.0, n[0] / 2 - 1.0]), steps=rng.randint(3, 20))
        if kind == "les":
            kw.update(sgs=rng.choice([0, 1, 1, 2]), forced=rng.choice([0, 1]))
            kw.update(scalar=kw["sgs"] == 0 or rng.random() < 0.5)
        return dns(*n, **kw)
    if kind in ("ens2d", "turb2d"):
        groups, room = [], 24 if kind == "ens2d" else 22
        for n in sorted(rng.sample([64, 128, 256, 512, 1024], rng.randint(1, 3))):
            most = max(1, (1 << room) // (n * n) // 3)
            groups.append((n, min(200, max(1, int(math.exp(rng.uniform(0, math.log(most + 1))))))))
        return ens(0 if kind == "ens2d" else 1, groups, steps=rng.randint(5, 50), eps=0.01 * eps)
    while True:
        n = [log_pow2(4, 7) for _ in range(3)]
        if 14 <= sum(a.bit_length() - 1 for a in n) <= 18:
            break
    steps = rng.randint(2, 20)
    return dict(kind="adjoint", nx=n[0], ny=n[1], nz=n[2], sgs=rng.choice([0, 1, 1]), steps=steps,
                ckpt=rng.randint(1, steps), nu=5e-3 * eps, dt=2e-3)


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def cut_of(c):
    """The truncation radius of a case's steps: 2/3 of nx/2 unless given."""
    return c.get("kcut") or 2.0 * (c["nx"] // 2) / 3.0


def waves(nx, ny, nz):
    kx = torch.arange(nx // 2 + 1, device=DEV, dtype=torch.float64)[None, None, :]
    ky = torch.fft.fftfreq(ny, 1.0 / ny, device=DEV, dtype=torch.float64)[None, :, None]
    kz = torch.fft.fftfreq(nz, 1.0 / nz, device=DEV, dtype=torch.float64)[:, None, None]
    return kx, ky, kz


def mirror(a):
    """conj a(-ky, -kz) of the kx = 0 plane of a half spectrum."""
    p = a[:, :, 0]
    return torch.roll(torch.flip(p, (0, 1)), (1, 1), (0, 1)).conj()


def zero_planes(a):
    nz, ny, lx1 = a.shape
    a[:, :, lx1 - 1] = 0
    a[:, ny // 2, :] = 0
    a[nz // 2, :, :] = 0
    a[0, 0, 0] = 0
    return a


def half_norm(f):
    """sum' |f|^2, half weight on kx = 0."""
    t = f.abs().square()
    return t.sum(dtype=torch.float64) - 0.5 * t[:, :, 0].sum(dtype=torch.float64)


def turbulent_field(c, seed, ncomp, k0=4.0):
    """ncomp half-spectrum fields (complex64 on the GPU) with a developed
    turbulence spectrum: E(k) ~ k^4 (1 + (k/k0)^2)^(-17/6) falling off towards
    the truncation radius, random phases, the three velocity components
    solenoidal, sum' |u|^2 = 1.5; zero beyond the truncation radius, as the
    solver's own states are."""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    gen = torch.Generator(DEV).manual_seed(int(seed) * 7919 + 17)
    kx, ky, kz = (a.float() for a in waves(nx, ny, nz))
    k2 = kx * kx + ky * ky + kz * kz
    kc = cut_of(c)
    shape = k2.clamp(min=1.0).sqrt() * (1 + k2 / k0**2) ** (-17.0 / 12.0) * torch.exp(-3.0 * k2 / kc**2)
    shape = torch.where(k2 >= kc * kc, torch.zeros_like(shape), shape)
    f = []
    for _ in range(ncomp):
        z = torch.randn((nz, ny, nx // 2 + 1), generator=gen, device=DEV, dtype=torch.complex64)
        z *= shape
        z[:, :, 0] = 0.5 * (z[:, :, 0] + mirror(z))
        f.append(zero_planes(z))
    if ncomp >= 3:
        q = (kx * f[0] + ky * f[1] + kz * f[2]) / k2.clamp(min=1.0)
        for a, k in zip(f, (kx, ky, kz)):
            a -= k * q
        del q
    norm = sum(half_norm(a) for a in f[:3])
    s = (1.5 / norm).sqrt().float()
    return [a * s for a in f]


def planar_field(n, members, seed, scheme):
    """Vorticity of `members` members, E(k) ~ k exp(-(k/8)^2) with a k^-3
    tail, random phases, enstrophy-carrying energy 0.5 each."""
    gen = torch.Generator(DEV).manual_seed(int(seed) * 104729 + 31 * n + scheme)
    kx = torch.arange(n // 2 + 1, device=DEV, dtype=torch.float32)[None, :]
    ky = torch.fft.fftfreq(n, 1.0 / n, device=DEV, dtype=torch.float32)[:, None]
    k2 = kx * kx + ky * ky
    kc = 2.0 * (n // 2) / 3.0
    k = k2.clamp(min=1.0).sqrt()
    shape = k * torch.exp(-k2 / 128.0) + 0.02 * k * (1 + k2 / 64.0) ** -2 * torch.exp(-4.0 * k2 / kc**2)
    shape = torch.where(k2 >= kc * kc, torch.zeros_like(shape), shape)
    w = torch.randn((members, n, n // 2 + 1), generator=gen, device=DEV, dtype=torch.complex64) * shape
    w[:, :, 0] = 0.5 * (w[:, :, 0] + torch.roll(torch.flip(w[:, :, 0], (1,)), 1, 1).conj())
    w[:, n // 2, :] = 0
    w[:, :, n // 2] = 0
    w[:, 0, 0] = 0
    e = w.abs().square() / k2.clamp(min=1.0)
    norm = e.sum((1, 2)) - 0.5 * e[:, :, 0].sum(1)
    return w * (0.5 / norm).sqrt()[:, None, None]


def ens_groups(c):
    return [tuple(int(x) for x in g.split("x")) for g in c["groups"].split()]


def ens_args(c):
    if c["scheme"]:
        big = max(n for n, _ in ens_groups(c))
        return dict(scheme=1, dt=1e-4, sigma=2.5 / big, nu=0.5, eta=5.0, kf=4.0)
    return dict(scheme=0, dt=5e-4, c_hyper=1e-5, n_hyper=8, damp=0.1, fkmin=4.0, fkmax=5.0, eps=c.get("eps", 0.01))


def dns_args(c):
    sgs = c["sgs"]
    return dict(nu=c["nu"], dt=c["dt"], forced=c["forced"], fkmax=2.5, eps=0.1, eta=0.2 if c["forced"] == 2 else 0.0,
                sgs=sgs, cs2=0.17**2 if sgs == 1 else 0.0, iupdate=10, scalar=c["scalar"],
                grad=1.0 if c["scalar"] else 0.0, schmidt=0.7, stepper=c["stepper"], beta=0.5, ieout=10,
                umax=3.0 * 3.0**0.5, kcut=c["kcut"])


def prec_of(c):
    return scl.SP if c.get("prec", "sp") == "sp" else scl.DP


def on_host(a, prec):
    return a.to(torch.complex64 if prec == scl.SP else torch.complex128).cpu().numpy()


class _Memory:
    """n complex entries at a device address, for torch to look at."""

    def __init__(self, ptr, n, prec):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<c8" if prec == scl.SP else "<c16",
                                             data=(ptr, False), version=2)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "ens2d":
        groups = ens_groups(c)
        e = scl.Ensemble2D(groups, prec=scl.SP, **ens_args(c))
        for g, (n, m) in enumerate(groups):
            w = planar_field(n, m, seed, c["scheme"])
            if c["scheme"]:  # wz(my, mx2): 2 conj of the normalised coefficients, no kx = n/2 column
                w = (2 * w.conj())[:, :, : n // 2].resolve_conj()
            w = w.cpu().numpy()
            for j in range(m):
                e.set_member(g, j, w[j])
        return dict(case=c, ens=e, groups=groups)
    prec = prec_of(c)
    plan = scl.Plan3D(c["nx"], c["ny"], c["nz"], prec)
    if kind == "dns":
        d = scl.DNS(plan, **dns_args(c))
        f = turbulent_field(c, seed, 4 if c["scalar"] else 3)
        d.set_velocity(*[on_host(a, prec) for a in f[:3]])
        if c["scalar"]:
            d.set_scalar(on_host(f[3], prec))
        ptr, n = d.state()
        v = torch.as_tensor(_Memory(ptr, n, prec), device=DEV)
        nc, rows = len(f), c["ny"] * c["nz"] * (c["nx"] // 2 + 1)
        fields = [v[q * (n // nc): q * (n // nc) + rows] for q in range(nc)]
        for a in fields:
            a.solver = d  # the memory is the solver's: it lives as long as the tensors handed out
        return dict(case=c, plan=plan, dns=d, fields=fields)
    if kind == "adjoint":
        a = scl.Adjoint(plan, c["steps"], c["ckpt"], nu=c["nu"], dt=c["dt"], sgs=c["sgs"])
        u0 = torch.stack(turbulent_field(c, seed, 3, 3.0))
        g = torch.stack(turbulent_field(c, seed + 1000, 3, 3.0))
        cs2 = torch.tensor(0.15**2 if c["sgs"] else 0.0, dtype=torch.float64, device=DEV)
        return dict(case=c, plan=plan, adj=a, u0=u0.requires_grad_(), cs2=cs2.requires_grad_(), gT=g)
    v = [on_host(a, prec) for a in turbulent_field(c, seed, 3)]
    return dict(case=c, plan=plan, v=v)


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "dns":
        state["dns"].step(c["steps"])
        return state["fields"]
    if kind == "ens2d":
        e = state["ens"]
        e.step(c["steps"])
        return [np.stack([e.get_member(g, j) for j in range(m)]) for g, (n, m) in enumerate(state["groups"])]
    if kind == "adjoint":
        uT = torch_adjoint.rk4_map(state["u0"], state["cs2"], state["adj"])
        g0, gc = torch.autograd.grad(uT, (state["u0"], state["cs2"]), state["gT"])
        return dict(uT=uT, g0=g0, gc=gc) if c["sgs"] else dict(uT=uT, g0=g0)
    return state["plan"].ratesdudt(*state["v"], forced=c["forced"], fkmax=2.5, eps=c.get("eps", 0.1), eta=0.2)


def work(case):
    """bytes: per step (per call for adjoint and rhs) the state read once and
    written once; flops: the real FFTs, 2.5 N log2 N each."""
    c, kind = case, case["kind"]
    if kind == "ens2d":
        pts = sum(m * n * n for n, m in ens_groups(c))
        fft = sum(2.5 * m * n * n * 2 * math.log2(n) for n, m in ens_groups(c))
        return dict(bytes=2.0 * 4 * pts * c["steps"], flops=c["steps"] * fft * (5 * 4 if c["scheme"] == 0 else 5 * 2))
    pts = c["nx"] * c["ny"] * c["nz"]
    fft = 2.5 * pts * math.log2(pts)
    es = 4 if c.get("prec", "sp") == "sp" else 8
    if kind == "rhs":
        return dict(bytes=6.0 * es * pts, flops=9 * fft)
    if kind == "adjoint":
        per = (9 + 12 * c["sgs"], 15 + 18 * c["sgs"])
        return dict(bytes=12.0 * es * pts, flops=4.0 * c["steps"] * (per[0] + per[1]) * fft)
    n = 9 + (12 if c["sgs"] else 0) + (4 if c["scalar"] else 0)
    stages = 1 if c["stepper"] else 4
    return dict(bytes=2.0 * es * pts * (4 if c["scalar"] else 3) * c["steps"], flops=c["steps"] * stages * n * fft)


# --------------------------------------------------------------------------
# The same passes in plain torch, FP64
# --------------------------------------------------------------------------
PAIRS = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]
TWICE = [1.0, 2.0, 2.0, 1.0, 2.0, 1.0]


class Spectral3D:
    """The pseudo-spectral RHS and steppers on half spectra (nz, ny, nx/2+1)."""

    def __init__(self, c):
        self.c = c
        self.n = c["nz"], c["ny"], c["nx"]
        self.k = waves(c["nx"], c["ny"], c["nz"])
        self.k2 = sum(a * a for a in self.k)
        self.inv_k2 = 1.0 / self.k2.clamp(min=1.0)
        self.keep = torch.ones_like(self.k2)
        zero_planes(self.keep)
        self.inside = (self.k2 < cut_of(c) ** 2).double()
        self.delta = 2 * math.pi / c["nx"]
        self.half = torch.full((c["nx"] // 2 + 1,), 1.0, device=DEV, dtype=torch.float64)
        self.half[0] = 0.5

    def phys(self, a):
        return torch.fft.irfftn(a, s=self.n, norm="forward")

    def spec(self, a):
        return torch.fft.rfftn(a, norm="forward")

    def strain(self, v, i, j):
        return 0.5j * (self.k[i] * v[j] + self.k[j] * v[i])

    def size(self, s):
        return torch.sqrt(2.0 * sum(w * a * a for w, a in zip(TWICE, s)))

    def curl(self, v):
        k = self.k
        return [1j * (k[(q + 1) % 3] * v[(q + 2) % 3] - k[(q + 2) % 3] * v[(q + 1) % 3]) for q in range(3)]

    def dynamic_cs2(self, v):
        g = (self.k2 <= (2.0 * (self.c["nx"] // 2) / 3.0 / 2.0) ** 2).double()
        u, ut = [self.phys(a) for a in v], [self.phys(g * a) for a in v]
        st = [self.phys(g * self.strain(v, i, j)) for i, j in PAIRS]
        s = [self.phys(self.strain(v, i, j)) for i, j in PAIRS]
        a, at = self.size(s), self.size(st)
        lm = mm = 0.0
        for q, (i, j) in enumerate(PAIRS):
            L = self.phys(g * self.spec(u[i] * u[j])) - ut[i] * ut[j]
            M = self.phys(g * self.spec(2 * self.delta**2 * a * s[q])) - 2 * (2 * self.delta) ** 2 * at * st[q]
            mm, lm = mm + TWICE[q] * (M * M).sum(), lm + TWICE[q] * (L * M).sum()
        return lm / mm

    def force(self, v, forced, eps, eta):
        band = (self.k2 < 2.5**2).double() * self.half

        def dot(a, b):
            return sum((band * (x.conj() * y).real).sum() for x, y in zip(a, b))

        w = self.curl(v)
        E, Om, uw = dot(v, v), dot(w, w), 2.0 * dot(v, w)
        a, b = eps / (2.0 * E), 0.0
        if forced == 2:
            den = 4.0 * E * Om - uw * uw
            a, b = (4.0 * eps * Om - eta * uw) / (2.0 * den), (eta * E - eps * uw) / den
        m = (self.k2 < 2.5**2).double()
        return [m * (a * x + b * y) for x, y in zip(v, w)]

    def rhs(self, y, forced, cs2=None, eps=0.1, eta=0.2):
        v = y[:3]
        u, w = [self.phys(a) for a in v], [self.phys(a) for a in self.curl(v)]
        n = [self.spec(u[(q + 1) % 3] * w[(q + 2) % 3] - u[(q + 2) % 3] * w[(q + 1) % 3]) for q in range(3)]
        del w
        if forced:
            n = [a + b for a, b in zip(n, self.force(v, forced, eps, eta))]
        if cs2 is not None:
            s = [self.phys(self.strain(v, i, j)) for i, j in PAIRS]
            # |S| with a zero gradient where S = 0
            m = 2.0 * sum(w_ * a * a for w_, a in zip(TWICE, s))
            size = torch.sqrt(m.clamp(min=1e-300))
            for q, (i, j) in enumerate(PAIRS):
                t = self.spec(-2.0 * cs2 * self.delta**2 * size * s[q])
                n[i] = n[i] - 1j * self.k[j] * t
                if i != j:
                    n[j] = n[j] - 1j * self.k[i] * t
        out = [self.sym(a) for a in n]
        q = sum(k * a for k, a in zip(self.k, out)) * self.inv_k2
        out = [a - k * q for k, a in zip(self.k, out)]
        if len(y) > 3:
            p = self.phys(y[3])
            r = -1j * sum(k * self.spec(a * p) for k, a in zip(self.k, u)) - y[2]
            out.append(self.sym(r))
        return out

    def sym(self, a):
        """The unpaired planes and the mean zeroed; on kx = 0 the modes with
        kz < 0, or kz = 0 and ky < 0, the conjugates of their partners."""
        a = a * self.keep
        nz, ny = a.shape[:2]
        src = torch.ones((nz, ny), device=DEV, dtype=torch.bool)
        src[nz // 2 + 1:, :] = False
        src[0, ny // 2 + 1:] = False
        plane = torch.where(src, a[:, :, 0], mirror(a))
        return torch.cat([plane[:, :, None], a[:, :, 1:]], 2)

    def rk4(self, y, dt, nus, forced, cs2=None):
        x = [-nu * self.k2 * dt / 2 for nu in nus]
        E = [torch.exp(a) for a in x]

        def N(s):
            return [dt * a for a in self.rhs(s, forced, cs2)]

        a1 = N(y)
        acc = [e * e * (v + a / 6) for e, v, a in zip(E, y, a1)]
        s = [e * (v + a / 2) for e, v, a in zip(E, y, a1)]
        del a1
        a2 = N(s)
        acc = [d + e * a / 3 for d, e, a in zip(acc, E, a2)]
        s = [e * v + a / 2 for e, v, a in zip(E, y, a2)]
        del a2
        a3 = N(s)
        acc = [d + e * a / 3 for d, e, a in zip(acc, E, a3)]
        s = [e * (e * v + a) for e, v, a in zip(E, y, a3)]
        del a3, y
        return [self.inside * (d + a / 6) for d, a in zip(acc, N(s))]

    def split(self, a):
        """The solver's device layout: rows of nx/2, then the kx = nx/2 plane;
        rows in blocks of 8 z for 1024-point z-lines."""
        nz, ny, lx1 = a.shape
        if nz >= 1024:
            a = a.reshape(nz // 8, 8, ny, lx1).transpose(1, 2)
        return torch.cat([a[..., : lx1 - 1].reshape(-1), a[..., lx1 - 1].reshape(-1)])


def exact_dns(c, seed):
    S = Spectral3D(c)
    y = [a.to(torch.complex128) for a in turbulent_field(c, seed, 4 if c["scalar"] else 3)]
    nus = [c["nu"]] * 3 + [c["nu"] / 0.7] * (len(y) - 3)
    cs2 = 0.17**2 if c["sgs"] == 1 else None
    if not c["stepper"]:
        for n in range(c["steps"]):
            if c["sgs"] == 2 and n % 10 == 0:
                cs2 = S.dynamic_cs2(y)
            y = S.rk4(y, c["dt"], nus, c["forced"], cs2)
        return [S.split(a) for a in y]
    inside = S.inside.clone()
    inside[0, 0, 0] = 0
    umax, dto, aux, n0 = 3.0 * 3.0**0.5, 1e30, None, None
    for n in range(c["steps"]):
        if c["stepper"] == 1:
            if n % 10 == 0:
                umax = 3.5 * math.sqrt(2.0 * float(sum(half_norm(a) for a in y[:3])))
            dt = min(0.5 * math.pi / (c["nx"] // 2) / umax, 3.0 * dto)
        else:
            dt = 0.5 * c["dt"] if n < 2 else c["dt"]
        N = S.rhs(y, c["forced"], cs2)
        E, r = torch.exp(-c["nu"] * S.k2 * dt), dt / dto
        Eo = torch.exp(-c["nu"] * S.k2 * dto) if n else None
        if n == 0:
            new, aux, n0, dto_new = [E * (v + dt * a) for v, a in zip(y, N)], y, N, dt
        elif n == 1:
            new = [E * (0.5 * (1 + r * r) * Eo * v0 + 0.5 * (1 - r * r) * v + 0.5 * dto * (1 + r) ** 2 * a)
                   for v0, v, a in zip(aux, y, N)]
            aux, dto_new = n0, dt + dto
        else:
            new = [E * (v + (1 + 0.5 * r) * dt * a - 0.5 * r * dt * Eo * o) for v, a, o in zip(y, N, aux)]
            aux, dto_new = N, dt
        y, dto = [inside * a for a in new], dto_new
    return [S.split(a) for a in y]


def exact_adjoint(c, seed):
    from torch.utils.checkpoint import checkpoint

    S = Spectral3D(c)
    u0 = torch.stack(turbulent_field(c, seed, 3, 3.0)).to(torch.complex128).requires_grad_()
    g = torch.stack(turbulent_field(c, seed + 1000, 3, 3.0)).to(torch.complex128)
    cs2 = torch.tensor(0.15**2, dtype=torch.float64, device=DEV, requires_grad=True)

    def step(u, cs):
        return torch.stack(S.rk4([u[0], u[1], u[2]], c["dt"], [c["nu"]] * 3, 0, cs if c["sgs"] else None))

    u = u0
    for _ in range(c["steps"]):
        u = checkpoint(step, u, cs2, use_reentrant=False)
    out = torch.autograd.grad(u, (u0, cs2) if c["sgs"] else (u0,), g)
    r = dict(uT=u.detach(), g0=out[0])
    if c["sgs"]:
        r["gc"] = out[1]
    return r


def exact_ens(c, seed):
    out, a = [], ens_args(c)
    for n, m in ens_groups(c):
        w = planar_field(n, m, seed, c["scheme"]).to(torch.complex128)
        kx = torch.arange(n // 2 + 1, device=DEV, dtype=torch.float64)[None, :]
        ky = torch.fft.fftfreq(n, 1.0 / n, device=DEV, dtype=torch.float64)[:, None]
        k2 = kx * kx + ky * ky
        ik2 = 1.0 / k2.clamp(min=1.0)
        k = k2.sqrt()
        keep = (k2 < ((2.0 * (n // 2) / 3.0) ** 2 if not c["scheme"] else 2.0 / 9.0 * n * n)).double()
        keep[n // 2, :] = 0
        keep[:, n // 2] = 0
        keep[0, 0] = 0

        def products(w):
            u, v, p = (torch.fft.irfft2(x, s=(n, n), norm="forward") for x in (1j * ky * ik2 * w, -1j * kx * ik2 * w, w))
            return [torch.fft.rfft2(x * p, norm="forward") for x in (u, v)]

        if not c["scheme"]:
            band = ((k2 >= 16.0) & (k2 <= 25.0)).double()
            rate, dt = a["c_hyper"] * k2**4 + a["damp"], a["dt"]

            def N(w):
                f, h = products(w)
                r = -1j * (kx * f + ky * h)
                r = r + a["eps"] * band * w / (w.abs().square() + 1e-300)
                return dt * keep * r

            E = torch.exp(-rate * dt / 2)
            cut = (k2 < (2.0 * (n // 2) / 3.0) ** 2).double()
            for _ in range(c["steps"]):
                a1 = N(w)
                a2 = N(E * (w + a1 / 2))
                a3 = N(E * w + a2 / 2)
                a4 = N(E * (E * w + a3))
                w = cut * (E * E * (w + a1 / 6) + E * (a2 + a3) / 3 + a4 / 6)
            out.append(w)
            continue
        ph = torch.exp(1j * math.pi / n * (kx + ky))
        lam = (k * a["sigma"]) ** 16 + (k2.clamp(min=0.5).sqrt() / a["nu"]) ** -4
        band = ((k >= 4.0) & (k <= 7.0)).double() * (a["eta"] / 104.0 / 4.0)
        dt = a["dt"]

        def N(w):
            f, h = products(w)
            fs, hs = products(w * ph.conj())
            return -0.5j * keep * (kx * f + ky * h + ph * (kx * fs + ky * hs))

        def F(x):
            return torch.where(band > 0, band * x / x.abs().square().clamp(min=1e-300), torch.zeros_like(x))

        E = torch.exp(-lam * dt)
        E[0, 0] = 1.0
        w0 = old = None
        for s in range(c["steps"]):
            r = N(w)
            if s == 0:
                w0, old, w = w, r, w * (1 - lam * dt / 2) + dt / 2 * (r + F(w))
            elif s == 1:
                w = w0 + dt * (r + F(w)) - lam * dt * w
            else:
                old, w = r, E * (w + dt / 2 * (3 * (r + F(w)) - E * (old + F(old))))
        out.append((2 * w.conj())[:, :, : n // 2].resolve_conj())
    return [x.cpu().numpy() for x in out]


def exact(case, seed):
    c = case
    if c["kind"] == "adjoint":
        return exact_adjoint(c, seed)
    with torch.no_grad():
        if c["kind"] == "dns":
            return exact_dns(c, seed)
        if c["kind"] == "ens2d":
            return exact_ens(c, seed)
        y = [a.to(torch.complex128) for a in turbulent_field(c, seed, 3)]
        return tuple(a.cpu().numpy() for a in Spectral3D(c).rhs(y, c["forced"], None, c.get("eps", 0.1), 0.2))
