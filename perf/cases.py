"""Timed cases of the solver: what a user of this framework has it do, through
its public entry points.

A case is one call (or one turn of a user's loop) of ``NS3D`` on a grid:

  step     ``RK3_SSP``: ``steps`` SSP-RK3 steps of one velocity field
  series   ``RK3_SSP`` and the energy and dissipation of the result (a time series)
  batch    ``RK3_SSP_batch``: ``members`` fields of one grid advanced together
  tangent  ``RK3_SSP_UV``: base flow and perturbation advanced by one step
  jv       ``jv_reduced``: one Jacobian-vector product of a Krylov solver
  scalar   ``RK3_SSP_scalar``: velocity steps with a WENO5 passive scalar

``precision`` is the context's ("fp64", or "fp32": FP32 transforms over an FP64
state); ``mode`` is "reference" (the reference's mask and IPQ rule, the default
of the library) or "physical" (IPQ off, 2/3 mask at the Nyquist wavenumbers: the
mode of the request server); ``forced`` adds the Kolmogorov forcing f_x = sin 4y.
Fields are the seeded solenoidal fields of the library's workloads
(E(k) ~ k^4 exp(-2 (k/4)^2), energy 0.5), made here on the GPU.
"""
import math

import numpy as np
import torch

from ns3dperiodic_amd import NS3D

SIZES = (16, 32, 48, 64, 80, 96, 128, 160, 192, 256, 320, 384, 512)
TWO_PI = 2.0 * math.pi


def _case(name, kind, nx, ny, nz, precision="fp64", mode="reference", forced=False, Re=100.0, steps=1, members=1,
          flow="random"):
    c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "precision": precision, "mode": mode, "forced": forced, "Re": Re,
         "steps": steps, "members": members, "flow": flow}
    return dict(c, name=name) if name else c


def listed():
    return [
        # The smallest call: one step of the 32^3 Shapiro exact-solution test, as a loop that looks at
        # the field after every step makes it; launches and latency are all there is.
        _case("shapiro_32_fp64", "step", 32, 32, 32, Re=20.0, flow="shapiro"),
        # A small uneven field of a parameter sweep: 20 steps to a call.
        _case("sweep_48x64x32_fp64", "step", 48, 64, 32, mode="physical", forced=True, steps=20),
        # Krylov work on a 64^3 Kolmogorov flow: one product with the Jacobian.
        _case("krylov_jv_64_fp64", "jv", 64, 64, 64, forced=True, Re=150.0),
        # 64 finite-difference perturbations of a 64^3 snapshot and the base flow, advanced together.
        _case("fd_batch_65x64_fp64", "batch", 64, 64, 64, mode="physical", forced=True, Re=150.0, members=65),
        # A served integrate request on a 96^3 grid (radix 3) in FP32 bulk: a chunk of 8 steps.
        _case("served_96_fp32", "step", 96, 96, 96, precision="fp32", mode="physical", forced=True, Re=200.0, steps=8),
        # Kolmogorov flow at 128^3 with energy and dissipation after every step.
        _case("series_128_fp64", "series", 128, 128, 128, mode="physical", forced=True, Re=100.0),
        # The tangent map (linear stability, Floquet multipliers) at 128^3.
        _case("tangent_128_fp64", "tangent", 128, 128, 128, Re=100.0),
        # A served integrate request on a 192^3 grid (radix 3), the one that most of the stream's time goes to.
        _case("served_192_fp64", "step", 192, 192, 192, mode="physical", forced=True, Re=200.0, steps=2),
        # Decaying turbulence at 256^3: the headline workload, in both precisions ...
        _case("turbulence_256_fp64", "step", 256, 256, 256, Re=500.0, steps=2),
        _case("turbulence_256_fp32", "step", 256, 256, 256, precision="fp32", Re=500.0, steps=2),
        # ... with a WENO5 passive scalar ...
        _case("scalar_256_fp64", "scalar", 256, 256, 256, Re=500.0),
        # ... and at 512^3, the largest grid.
        _case("turbulence_512_fp64", "step", 512, 512, 512, Re=500.0),
    ]


def draw(rng):
    """One more case of the ranges above: any grid the library has plans for, its axes within a factor of two of
    each other, sizes spread over their logarithm."""
    kind = rng.choice(("step", "step", "step", "step", "series", "batch", "tangent", "jv", "scalar"))
    top = {"step": 512, "series": 384, "batch": 96, "tangent": 256, "jv": 256, "scalar": 320}[kind]
    low = {"scalar": 32, "series": 32}.get(kind, 16)
    want = math.exp(rng.uniform(math.log(low), math.log(top)))
    base = min((n for n in SIZES if n <= top), key=lambda n: abs(math.log(n / want)))
    n = [base if rng.random() < 0.4 else rng.choice([s for s in SIZES if base / 2 <= s <= min(2 * base, top)])
         for _ in range(3)]
    points = n[0] * n[1] * n[2]
    members = 1
    if kind == "batch":
        members = max(2, min(96, int(math.exp(rng.uniform(math.log(2), math.log(2 ** 25 / points))))))
    steps = 1
    if kind in ("step", "scalar"):
        steps = rng.choice((1, 2, 3, 5, 8, 20)) if points <= 64 ** 3 else rng.choice((1, 2, 3)) if points <= 192 ** 3 else 1
    # the library's reference mode on large decaying or Krylov work, the physical mode on forced flows
    mode = rng.choice(("reference", "physical")) if points >= 96 ** 3 or kind in ("jv", "tangent") else "physical"
    return _case(None, kind, n[0], n[1], n[2], precision=rng.choice(("fp64", "fp64", "fp32")) if kind != "jv" else "fp64",
                 mode=mode, forced=mode == "physical" and rng.random() < 0.6, Re=round(rng.uniform(60.0, 500.0), 1),
                 steps=steps, members=members)


# ---------------------------------------------------------------- inputs
def _dt(case):
    """CFL 0.2 at max |u| = 2.6, the bench's choice at 256^3; 1e-3 for the Shapiro test."""
    if case["flow"] == "shapiro":
        return 1.0e-3
    return 0.2 * TWO_PI / max(case["nx"], case["ny"], case["nz"]) / 2.6


def _wavenumbers(nx, ny, nz, device):
    def full(n):
        m = torch.arange(n, device=device, dtype=torch.float64)
        return torch.where(m >= n // 2, m - n, m)
    kz = torch.arange(nz // 2 + 1, device=device, dtype=torch.float64)
    return full(nx).view(-1, 1, 1), full(ny).view(1, -1, 1), kz.view(1, 1, -1)


def _random_solenoidal(nx, ny, nz, gen, device):
    """Three spectral fields of one seeded divergence-free field, energy 0.5."""
    kx, ky, kz = _wavenumbers(nx, ny, nz, device)
    k2 = kx * kx + ky * ky + kz * kz
    safe = torch.where(k2 == 0, 1.0, k2)
    amp = safe.sqrt() * torch.exp(-safe / 16.0)  # sqrt(E(k) / k^2)
    amp[nx // 2, :, :] = 0
    amp[:, ny // 2, :] = 0
    amp[:, :, nz // 2] = 0
    amp[0, 0, 0] = 0
    u = [torch.fft.rfftn(torch.randn((nx, ny, nz), generator=gen, device=device, dtype=torch.float64)) * amp
         for _ in range(3)]
    kd = (kx * u[0] + ky * u[1] + kz * u[2]) / safe
    u = [u[0] - kx * kd, u[1] - ky * kd, u[2] - kz * kd]
    w = torch.full((nz // 2 + 1,), 2.0, device=device, dtype=torch.float64)
    w[0] = w[-1] = 1.0
    n3 = float(nx) * ny * nz
    e = sum(float(((c.real ** 2 + c.imag ** 2) * w).sum()) for c in u) / (n3 * n3)
    s = math.sqrt(1.0 / e)                   # mean |u|^2 = 1: energy 0.5
    return [(c * s).contiguous() for c in u]


def _shapiro(nx, ny, nz, seed, device):
    """The Shapiro Beltrami field at t = 0, moved in x by a seeded phase (a solution again)."""
    x, y, z = [(torch.arange(n, device=device, dtype=torch.float64) * (TWO_PI / n)) for n in (nx, ny, nz)]
    x = x.view(-1, 1, 1) + 0.1 * (seed % 61)
    y, z = y.view(1, -1, 1), z.view(1, 1, -1)
    f = math.sqrt(3.0)
    ux = -0.5 * (f * torch.cos(x) * torch.sin(y) * torch.sin(z) + torch.sin(x) * torch.cos(y) * torch.cos(z))
    uy = 0.5 * (f * torch.sin(x) * torch.cos(y) * torch.sin(z) - torch.cos(x) * torch.sin(y) * torch.cos(z))
    uz = torch.cos(x) * torch.cos(y) * torch.sin(z)
    return [torch.fft.rfftn(c).contiguous() for c in (ux, uy, uz)]


def _forcing(nx, ny, nz, device):
    """f_x = sin 4y, as the reference's spectral arrays hold it."""
    f = [torch.zeros((nx, ny, nz // 2 + 1), dtype=torch.complex128, device=device) for _ in range(3)]
    n3 = float(nx) * ny * nz
    f[0][0, 4, 0] = -0.5j * n3
    f[0][0, ny - 4, 0] = 0.5j * n3
    return f


def _inputs(case, seed):
    device = torch.device("cuda", 0)
    shape = case["nx"], case["ny"], case["nz"]
    gen = torch.Generator(device=device)
    gen.manual_seed(int(seed))
    s = {"f": _forcing(*shape, device) if case["forced"] else None}
    if case["kind"] == "batch":
        # a base flow and seeded unit-norm perturbations of it, scaled by 1e-7 of its norm
        base = _random_solenoidal(*shape, gen, device)
        norm = math.sqrt(sum(float((c.real ** 2 + c.imag ** 2).sum()) for c in base))
        ub = torch.empty((case["members"], 3) + tuple(base[0].shape), dtype=torch.complex128, device=device)
        for m in range(case["members"]):
            p = _random_solenoidal(*shape, gen, device) if m else base
            size = math.sqrt(sum(float((c.real ** 2 + c.imag ** 2).sum()) for c in p))
            for b in range(3):
                ub[m, b] = base[b] + p[b] * (1e-7 * norm / size) if m else base[b]
        s["u"] = ub
        return s
    s["u"] = _shapiro(*shape, int(seed), device) if case["flow"] == "shapiro" else _random_solenoidal(*shape, gen, device)
    if case["kind"] == "tangent":
        s["v"] = [1e-3 * c for c in _random_solenoidal(*shape, gen, device)]
    elif case["kind"] == "jv":
        v = _random_solenoidal(*shape, gen, device)
        vec = torch.cat([c.imag.reshape(-1)[1:] for c in v])
        s["vec"] = vec / torch.linalg.vector_norm(vec)
    elif case["kind"] == "scalar":
        # a Gaussian random scalar of unit variance, E(k) ~ k^2 exp(-(k/4)^2)
        kx, ky, kz = _wavenumbers(*shape, device)
        amp = torch.exp(-(kx * kx + ky * ky + kz * kz) / 32.0)
        amp[0, 0, 0] = 0
        noise = torch.fft.rfftn(torch.randn(shape, generator=gen, device=device, dtype=torch.float64))
        th = torch.fft.irfftn(noise * amp, s=shape)
        s["theta"] = (th / th.std()).contiguous()
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    physical = case["mode"] == "physical"
    g = NS3D(case["nx"], case["ny"], case["nz"], Re=case["Re"], dt=_dt(case), precision=case["precision"],
             ipq=not physical, mask_nyquist=physical)
    s.update(g=g, kind=case["kind"], steps=case["steps"])
    if case["kind"] == "jv":
        g.set_base_state(s["u"], s["f"])
    return s


def run(s):
    g, kind = s["g"], s["kind"]
    if kind == "step":
        return g.RK3_SSP(s["u"], s["f"], steps=s["steps"])
    if kind == "series":
        u = g.RK3_SSP(s["u"], s["f"], steps=s["steps"])
        return [u, g.kinetic_energy_spectral(u), g.dissipation_spectral(u)]
    if kind == "batch":
        return g.RK3_SSP_batch(s["u"], s["f"], steps=s["steps"])
    if kind == "tangent":
        return g.RK3_SSP_UV(s["u"], s["v"], s["f"])
    if kind == "jv":
        return g.jv_reduced(s["vec"])
    u, theta = g.RK3_SSP_scalar(s["u"], s["theta"], s["f"], steps=s["steps"])
    return [u, theta]


# ---------------------------------------------------------------- work
def work(case):
    """Inputs read once, outputs written once; the transforms and pointwise arithmetic of the method:
    a velocity stage is 12 inverse and 3 forward real 3D transforms, a bilinear stage 24 and 3."""
    n3 = float(case["nx"]) * case["ny"] * case["nz"]
    nc = float(case["nx"]) * case["ny"] * (case["nz"] // 2 + 1)
    fft = 2.5 * n3 * math.log2(n3)
    stage = 15 * fft + 15 * n3 + 100 * nc
    bilinear = 27 * fft + 30 * n3 + 100 * nc
    field = 16 * nc
    forcing = 3 * field if case["forced"] else 0
    kind = case["kind"]
    if kind == "jv":
        return {"bytes": 3 * field + 2 * 24 * (nc - 1), "flops": bilinear}
    if kind == "tangent":
        return {"bytes": 12 * field + forcing, "flops": 3 * stage + 2 * bilinear + 30 * nc}
    flops = case["members"] * case["steps"] * 3 * stage
    byts = case["members"] * 6 * field + forcing
    if kind == "scalar":  # a WENO5 stage: six faces of about 60 operations to a point
        return {"bytes": byts + 16 * n3, "flops": flops + case["steps"] * 3 * 400 * n3}
    return {"bytes": byts, "flops": flops + (40 * nc if kind == "series" else 0)}


# ---------------------------------------------------------------- the same in plain torch, 64 bits
class _Exact:
    """The method in torch: spectral fields [..., Nx, Ny, Nz/2+1], unnormalised forward transforms."""

    def __init__(self, case, device):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        self.shape, self.dt, self.Re = (nx, ny, nz), _dt(case), case["Re"]
        self.k = _wavenumbers(nx, ny, nz, device)
        kx, ky, kz = self.k
        self.k2 = kx * kx + ky * ky + kz * kz
        self.ipq = case["mode"] == "reference"
        # the reference's 2/3 mask is relative to (Nx, Ny, Nz/2+1), the physical one to the Nyquist wavenumbers
        # (on the host, in the operations' own order: modes on the boundary go by its rounding)
        top = [2 * n * math.pi / TWO_PI for n in (nx, ny, nz // 2 + 1)] if self.ipq else [
            n * math.pi / TWO_PI for n in (nx, ny, nz)]
        part = [k.cpu().numpy() * 2 * math.pi / TWO_PI for k in self.k]
        mx, my, mz = [k * k / (t * t) for k, t in zip(part, top)]
        mask = (np.sqrt(mx + my + mz) < 2.0 / 3.0).astype(np.float64)
        mask[0, 0, 0] = 0.0
        self.mask = torch.from_numpy(mask).to(device)

    def real(self, c):
        """Inverse transform: x and y complex, then z from the half spectrum (real parts of its end planes)."""
        c = torch.fft.ifftn(c, dim=(-3, -2))
        c[..., 0].imag.zero_()
        c[..., -1].imag.zero_()
        return torch.fft.irfft(c, n=self.shape[2], dim=-1)

    def spec(self, r):
        return torch.fft.fftn(torch.fft.rfft(r, dim=-1), dim=(-3, -2))

    def gradients(self, c):
        c = c * self.mask
        return self.real(c), [self.real(1j * k * c) for k in self.k]

    def advect(self, u, v=None):
        """(u.grad)u, or with v (v.grad)u + (u.grad)v, in spectral space under the mode's rule for its real part."""
        phys = [self.real(c * self.mask) for c in u]
        vp = None if v is None else [self.real(c * self.mask) for c in v]
        out = []
        for b in range(3):
            du = self.gradients(u[b])[1]
            q = sum((phys if v is None else vp)[a] * du[a] for a in range(3))
            if v is not None:
                dv = self.gradients(v[b])[1]
                q = q + sum(phys[a] * dv[a] for a in range(3))
            q = self.spec(q)
            if self.ipq:
                q.real.zero_()
                q[..., 0, 0, 0] = 0
            out.append(q)
        return out

    def project(self, q):
        """A Q - Q with A = k k^T / |k|^2 (0 at k = 0)."""
        safe = torch.where(self.k2 == 0, 1.0, self.k2)
        kd = sum(k * c for k, c in zip(self.k, q)) / safe
        return [k * kd - c for k, c in zip(self.k, q)]

    def rhs(self, u, f=None, v=None):
        r = self.project(self.advect(u, v))
        w = u if v is None else v
        r = [a - self.k2 / self.Re * c for a, c in zip(r, w)]
        return r if f is None else [a + b for a, b in zip(r, f)]

    def euler(self, u, f=None, v=None):
        w = u if v is None else v
        return [c + self.dt * a for c, a in zip(w, self.rhs(u, f, v))]

    def rk3(self, u, f):
        a = self.euler(u, f)
        a = [0.75 * c + 0.25 * d for c, d in zip(u, self.euler(a, f))]
        return [c / 3.0 + d * (2.0 / 3.0) for c, d in zip(u, self.euler(a, f))]

    def scalar_euler(self, u, th):
        vel = [self.real(c * self.mask) for c in u]
        adv = 0
        for axis in range(3):
            adv = adv + vel[axis] * (self.shape[axis] / TWO_PI) * self.weno_difference(vel[axis], th, axis)
        return th - self.dt * adv

    @staticmethod
    def weno_difference(vel, th, axis):
        """Upwind WENO5 face values at +1/2 less those at -1/2 along an axis."""
        def at(f, o):
            return torch.roll(f, -o, dims=axis)

        def weno5(a, b, c, d, e):
            q = (a / 3 - 7 * b / 6 + 11 * c / 6, -b / 6 + 5 * c / 6 + d / 3, c / 3 + 5 * d / 6 - e / 6)
            s = (13 / 12 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2,
                 13 / 12 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2,
                 13 / 12 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2)
            w = [g / (1e-22 + x) ** 2 for g, x in zip((0.1, 0.6, 0.3), s)]
            return (w[0] * q[0] + w[1] * q[1] + w[2] * q[2]) / (w[0] + w[1] + w[2])

        face = 0.5 * (vel + at(vel, 1))  # velocity at +1/2
        left = weno5(at(th, -2), at(th, -1), th, at(th, 1), at(th, 2))
        # the reference's z reconstruction from the right ends at offset 0 where the stencil has -1
        right = weno5(at(th, 3), at(th, 2), at(th, 1), th, th if axis == 2 else at(th, -1))
        value = torch.where(face >= 0, left, right)
        return value - at(value, -1)


def exact(case, seed):
    s = _inputs(case, seed)
    x = _Exact(case, torch.device("cuda", 0))
    kind, f = case["kind"], s["f"]
    if kind == "jv":
        nc = case["nx"] * case["ny"] * (case["nz"] // 2 + 1)
        v = []
        for part in s["vec"].split(nc - 1):
            c = torch.zeros(nc, dtype=torch.complex128, device=part.device)
            c[1:] = 1j * part
            v.append(c.view(s["u"][0].shape))
        return torch.cat([c.imag.reshape(-1)[1:] for c in x.rhs(s["u"], None, v)])
    if kind == "batch":
        u = [s["u"][:, b].contiguous() for b in range(3)]
        for _ in range(case["steps"]):
            u = x.rk3(u, f)
        return torch.stack(u, dim=1)
    if kind == "tangent":
        u, v = s["u"], s["v"]
        a = x.euler(u, None, v)
        u = x.rk3(u, f)
        a = x.euler(u, None, a)
        return u, [0.5 * c + 0.5 * d for c, d in zip(v, a)]
    u, th = s["u"], s.get("theta")
    for _ in range(case["steps"]):
        if th is not None:
            u1 = x.euler(u, f)
            u2 = [0.75 * c + 0.25 * d for c, d in zip(u, x.euler(u1, f))]
            t1 = x.scalar_euler(u, th)
            t2 = 0.75 * th + 0.25 * x.scalar_euler(u1, t1)
            th = th / 3.0 + x.scalar_euler(u2, t2) * (2.0 / 3.0)
        u = x.rk3(u, f)
    if kind == "scalar":
        return [u, th]
    if kind == "series":
        n3 = float(np.prod(x.shape))
        w = torch.full((x.shape[2] // 2 + 1,), 2.0, device=u[0].device, dtype=torch.float64)
        w[0] = w[-1] = 1.0
        e = w * sum(c.real ** 2 + c.imag ** 2 for c in u)
        kd = sum(k * c for k, c in zip(x.k, u))
        volume = TWO_PI ** 3 / (n3 * n3)
        return [u, 0.5 * volume * float(e.sum()),
                volume * float((x.k2 * e + w * (kd.real ** 2 + kd.imag ** 2)).sum())]
    return u
