"""Workloads of the steppers as a program calls them, for timing and comparison.

A pass of a "run" case restarts every member from a snapshot held on the GPU
(a zero-copy view of the context's state, written on the context's stream) and
advances it `steps` time steps with Stepper.run(): one flow map of a Newton
solver, one output block of a DNS.  "tangent" is the Newton solver's Jv (one
base flow, several perturbations about it), "adjoint" the gradient sweep; both
are called on host arrays, as their entry points take them.

An FP64 case returns the state itself, an FP32-bulk case the single-precision
snapshot that a program keeps of a run whose transforms are single precision.
The states are broadband: solenoidal vorticity with E(k) ~ k^-5/3 and energy
0.5 over every active mode, as a developed flow has it.
"""
import math

import numpy as np
import torch

import psgpu_amd as P

FIELDS = {"ns2d": 1, "ns3d": 3, "euler": 3, "bous": 4}


def case(name, kind, flavour, nx, ny, nz, steps, precision="fp64", batch=1, extra=0, diag=False):
    c = dict(kind=kind, flavour=flavour, nx=nx, ny=ny, nz=nz, steps=steps, precision=precision, batch=batch,
             extra=extra, diag=diag)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest flow of a 2D Newton solve: launches and latency
        case("ns2d_128_run60", "run", "ns2d", 128, 128, 1, 60),
        # the 2D Kolmogorov flow the orbits are searched in: one flow map of its solver
        case("ns2d_512_run40", "run", "ns2d", 512, 512, 1, 40),
        # many Newton guesses on the members of one context
        case("ns2d_512_x8_run20", "run", "ns2d", 512, 512, 1, 20, batch=8),
        # tangent-linear Jv of two directions about one base flow
        case("ns2d_512_tangent", "tangent", "ns2d", 512, 512, 1, 20, extra=2),
        # the smallest 3D flow of use (minimal boxes of 3D orbits)
        case("ns3d_64_run50", "run", "ns3d", 64, 64, 64, 50),
        # an output block of a 128^3 DNS: the steps between two outputs, then the diagnostics
        case("ns3d_128_block50", "run", "ns3d", 128, 128, 128, 50, diag=True),
        # the benchmark's flow, FP64 and FP32-bulk
        case("ns3d_256_run20", "run", "ns3d", 256, 256, 256, 20),
        case("ns3d_256_fp32_run20", "run", "ns3d", 256, 256, 256, 20, precision="fp32"),
        # an ensemble in an elongated box: unequal extents, odd counts
        case("euler_256x128x64_x3_run7", "run", "euler", 256, 128, 64, 7, batch=3),
        # gradient of a flow with respect to its initial state
        case("ns3d_128_adjoint20", "adjoint", "ns3d", 128, 128, 128, 20, extra=10),
        # stratified ensemble in FP32-bulk, and the largest single flow
        case("bous_256_fp32_x2_run3", "run", "bous", 256, 256, 256, 3, precision="fp32", batch=2),
        case("bous_512_run1", "run", "bous", 512, 512, 512, 1),
    ]


def rhs_count(c):
    return {"ns2d": 4, "ns3d": 2, "euler": 2, "bous": 4}[c["flavour"]] * c["steps"] * c["batch"]


def points(c):
    return c["nx"] * c["ny"] * c["nz"]


def draw(rng):
    """One more case of the same ranges: 2D 64..1024, 3D 32..256 (and single 512^3 steps),
    each extent by itself, any step count, ensembles, both precisions."""
    kind = rng.choice(["run"] * 8 + ["tangent", "adjoint"])
    flavour = {"tangent": "ns2d", "adjoint": "ns3d"}.get(kind) or rng.choice(["ns2d", "ns2d", "ns3d", "ns3d", "ns3d",
                                                                              "euler", "bous"])
    precision = "fp64" if kind != "run" else rng.choice(["fp64", "fp64", "fp32"])
    batch, extra = 1, 0
    if flavour == "ns2d":
        ny = rng.choice([64, 128, 256, 512, 1024])
        nx, nz = rng.choice([ny, ny, ny // 2 if ny > 64 else ny, 2 * ny if ny < 1024 else ny]), 1
        steps = rng.randint(1, 60)
        if kind == "run":
            batch = rng.choice([1, 1, rng.randint(2, 16)])
        else:
            extra, steps = rng.randint(1, 4), rng.randint(5, 40)
    else:
        if kind == "run" and rng.random() < 0.1:
            nx = ny = nz = 512
            steps = 1
        else:
            ny = rng.choice([32, 64, 64, 128, 128, 256])
            side = lambda: rng.choice([ny, ny, ny, max(32, ny // 2), min(256, 2 * ny)])
            nx, nz = side(), side()
            steps = rng.randint(1, 60) if ny < 256 else rng.randint(1, 12)
            if kind == "run":
                batch = rng.choice([1, 1, rng.randint(2, 5)])
            else:
                nx, nz, steps = min(nx, 128), min(nz, 128), rng.randint(2, 24)
                ny = min(ny, 128)
                extra = rng.randint(2, max(2, steps))
    c = case(None, kind, flavour, nx, ny, nz, steps, precision, batch, extra, kind == "run" and rng.random() < 0.2)
    most = 4 * 512 ** 3     # grid points times right-hand sides of the largest listed case
    c["steps"] = max(1, min(steps, int(steps * most / max(most, points(c) * rhs_count(c)))))
    return c


# ------------------------------------------------------------------ grid
class Modes:
    """Wavenumbers, active mask and padded positions of the stored modes, on the GPU in FP64."""

    def __init__(self, c):
        self.two = c["flavour"] == "ns2d"
        self.n = (c["nz"], c["ny"], c["nx"])
        ktz, kty, ktx = (0 if self.two else c["nz"] // 3), c["ny"] // 3, c["nx"] // 3
        self.shape = (2 * ktz + 1, 2 * kty + 1, ktx + 1)
        self.alpha = c["ny"] / c["nx"]
        d = dict(dtype=torch.float64, device="cuda")
        self.kx = (torch.arange(ktx + 1, **d) * self.alpha)[None, None, :]
        self.ky = torch.arange(-kty, kty + 1, **d)[None, :, None]
        self.kz = torch.arange(-ktz, ktz + 1, **d)[:, None, None]
        self.k2 = self.kx ** 2 + self.ky ** 2 + self.kz ** 2
        self.ki = 1.0 / torch.clamp(self.k2, min=1e-3)
        half = (self.kx > 0) | ((self.kx == 0) & (self.ky > 0)) | ((self.kx == 0) & (self.ky == 0) & (self.kz > 0))
        self.L = (half & (self.k2.sqrt() <= kty - 0.5)).to(torch.float64)
        self.mirror = (self.ky < 0) | ((self.ky == 0) & (self.kz < 0))       # of the kx = 0 plane
        self.origin = (self.ky == 0) & (self.kz == 0)
        self.yi = torch.arange(-kty, kty + 1, device="cuda") % c["ny"]
        self.zi = torch.arange(-ktz, ktz + 1, device="cuda") % c["nz"]

    def fill(self, s):
        """The kx = 0 plane made Hermitian from its stored half."""
        p = s[..., :1]
        q = torch.where(self.mirror, p.flip(-3, -2).conj(), p) * (~self.origin)
        return torch.cat([q, s[..., 1:]], dim=-1)

    def grid(self, s):
        nz, ny, nx = self.n
        a = torch.zeros(s.shape[:-3] + (nz, ny, nx // 2 + 1), dtype=s.dtype, device=s.device)
        a[..., self.zi[:, None], self.yi[None, :], :self.shape[2]] = s
        return torch.fft.irfftn(a, s=self.n, dim=(-3, -2, -1), norm="forward")

    def modes(self, r):
        a = torch.fft.rfftn(r, dim=(-3, -2, -1), norm="forward")
        return a[..., self.zi[:, None], self.yi[None, :], :self.shape[2]]

    def curl(self, a, b, c):
        kx, ky, kz = self.kx, self.ky, self.kz
        return 1j * (ky * c - kz * b), 1j * (kz * a - kx * c), 1j * (kx * b - ky * a)


def physics(c):
    """Keyword arguments of the context: Re and dt in the range of the grid."""
    kw = dict(flavour=c["flavour"], nx=c["nx"], ny=c["ny"], nz=c["nz"], n=c["ny"], alpha=c["ny"] / c["nx"],
              batch=c["batch"], precision=c["precision"], force="kolmogorov", kf=4.0)
    if c["flavour"] == "ns2d":
        kw.update(v2=1 / 40.0, dt=min(0.005, 1.0 / c["ny"]), ampfor=-2.0)
    else:
        kw.update(v2=1 / 100.0 if c["flavour"] != "bous" else 1 / 400.0, dt=0.4 / max(c["ny"], 128))
        if c["flavour"] == "euler":
            kw.update(force="none")
        if c["flavour"] == "bous":
            kw.update(ri=1.0, sc=1.0, theta=90.0)
    return kw


def states(c, seed, count, energy=0.5):
    """`count` random states [count, nf, nkt] of the case's grid, from the seed alone."""
    m = Modes(c)
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = m.k2.sqrt()
    amp = m.L * (1 + (k / 4) ** 2) ** (-11 / 12 if not m.two else -2 / 3) * torch.exp(-2 * k / (c["ny"] / 3))
    out = torch.zeros((count, FIELDS[c["flavour"]]) + m.shape, dtype=torch.complex128, device="cuda")
    noise = lambda: torch.view_as_complex(torch.randn(m.shape + (2,), generator=g, dtype=torch.float64, device="cuda"))
    for i in range(count):
        if m.two:
            out[i, 0] = amp * k * noise()
        else:
            u = [amp * noise() for _ in range(3)]
            for f, w in enumerate(m.curl(*u)):
                out[i, f] = w
            del u
        s = math.sqrt(energy / float((out[i, :3].abs() ** 2 * m.ki).sum()))
        out[i, :3] *= s
        if c["flavour"] == "bous":
            r = amp * noise()
            out[i, 3] = r * (0.1 / float((r.abs() ** 2).sum())) ** 0.5
    return out.reshape(count, FIELDS[c["flavour"]], -1)


class StateArray:
    """A context's states as a tensor can view them; the view keeps the context, which owns the memory."""

    def __init__(self, stepper, shape):
        self.owner = stepper
        self.__cuda_array_interface__ = {"data": (stepper.state_ptr(0), False), "shape": shape, "typestr": "<c16",
                                         "version": 3}


def view_states(stepper, shape):
    t = torch.as_tensor(StateArray(stepper, shape), device="cuda")
    t.owner = stepper       # the returned tensor outlives the pass that it comes from
    return t


# ------------------------------------------------------------------ one pass
def prepare(case, seed):
    c = case
    kw = physics(c)
    s = {"case": c, "stepper": P.Stepper(**kw)}
    if c["kind"] == "run":
        st = s["stepper"]
        s["start"] = states(c, seed, c["batch"])
        s["stream"] = torch.cuda.ExternalStream(P.lib().psg_stream(st.h))
        s["field"] = view_states(st, tuple(s["start"].shape))
        if c["precision"] == "fp32":
            s["snapshot"] = torch.zeros(s["start"].shape, dtype=torch.complex64, device="cuda")
    else:
        z = states(c, seed, 1 + max(1, c["extra"] if c["kind"] == "tangent" else 1)).cpu().numpy()
        s["z"], s["d"] = z[0], z[1:]
    torch.cuda.synchronize()
    return s


def run(state):
    c, st = state["case"], state["stepper"]
    if c["kind"] == "tangent":
        dt = st.cfg.dt
        z, d = st.tangent_many(state["z"], state["d"], span(c, physics(c)["dt"]), physics(c)["dt"])
        return {"flow": z, "jv": d}
    if c["kind"] == "adjoint":
        z, lam = st.adjoint(state["z"], state["d"][0], c["steps"], c["extra"])
        return {"flow": z, "gradient": lam}
    with torch.cuda.stream(state["stream"]):
        state["field"].copy_(state["start"])
        st.run(c["steps"])
        out = {"state": state["field"]}
        if c["precision"] == "fp32":
            out["state"] = state["snapshot"].copy_(state["field"])
    if c["diag"]:
        energy, enstrophy, spectrum = st.diag()
        if c["precision"] == "fp32":
            spectrum = spectrum.astype(np.float32)
            energy, enstrophy = np.float32(energy), np.float32(enstrophy)
        out.update(energy=energy, enstrophy=enstrophy, spectrum=spectrum)
    return out


def span(c, dt):
    """A period of `steps` steps a little longer than dt, as the solver's time policy cuts it."""
    return (c["steps"] + 0.25) * dt


def work(case):
    """Every right-hand side reads the state and writes it; its real transforms are 2.5 N log2 N each."""
    c = case
    iky, ikz = 2 * (c["ny"] // 3) + 1, (2 * (c["nz"] // 3) + 1 if c["nz"] > 1 else 1)
    nkt = (c["nx"] // 3 + 1) * iky * ikz
    fields = {"ns2d": 3 + 2, "ns3d": 6 + 3, "euler": 6 + 3, "bous": 9 + 4}[c["flavour"]]
    real = 8 if c["precision"] == "fp64" else 4
    rhs = rhs_count(c)
    if c["kind"] == "tangent":
        rhs *= 1 + c["extra"]        # the base, and each direction about it
    n = points(c)
    flops = rhs * fields * 2.5 * n * math.log2(n)
    moved = rhs * 2 * FIELDS[c["flavour"]] * nkt * 2 * real
    if c["kind"] == "adjoint":
        flops *= 1 + 15 / 9          # forward, and the transposed steps' nine and six transforms
        moved *= 2
    return {"bytes": float(moved), "flops": float(flops)}


# ------------------------------------------------------------------ the same in 64 bits with torch alone
class Flow:
    def __init__(self, c, dt=None):
        self.m, self.kw, self.fl = Modes(c), physics(c), c["flavour"]
        self.dt = dt or self.kw["dt"]

    def product2(self, z, d=None):
        """-i k . FFT(u z), or its derivative along d."""
        m = self.m
        phys = lambda a: (m.grid(a), m.grid(1j * m.ky * m.ki * a), m.grid(-1j * m.kx * m.ki * a))
        w, u, v = phys(m.fill(z))
        if d is None:
            uw, vw = u * w, v * w
        else:
            dw, du, dv = phys(m.fill(d))
            uw, vw = du * w + u * dw, dv * w + v * dw
        return -1j * (m.kx * m.modes(uw) + m.ky * m.modes(vw))

    def step2(self, z, d=None):
        m, dt, nu = self.m, self.dt, self.kw["v2"]
        F = self.kw["ampfor"] * ((m.kx == 0) & (m.ky.abs() == self.kw["kf"]))
        parts = [z * m.L] + ([] if d is None else [d * m.L])
        first, acc = list(parts), [0] * len(parts)
        for weight, frac in ((1, 0.5), (2, 0.5), (2, 1.0), (1, None)):
            inc = [dt * m.L * (self.product2(parts[0]) + F)]
            if d is not None:
                inc.append(dt * m.L * self.product2(*parts))
            for i, x in enumerate(inc):
                acc[i] = acc[i] + weight * x
                parts[i] = first[i] + frac * x if frac else None
        half = 0.5 * dt * nu * m.k2
        done = [m.L * ((1 - half) * a + b / 6) / (1 + half) for a, b in zip(first, acc)]
        return done[0] if d is None else done

    def rhs3(self, w):
        """i k x FFT(u x w) of a state [3, ...] already filled."""
        m = self.m
        w = m.fill(w)
        x = [m.grid(a) for a in w]
        u = [m.grid(a * m.ki) for a in m.curl(*w)]
        cross = lambda i, j: m.modes(u[i] * x[j] - u[j] * x[i])
        return torch.stack(m.curl(cross(1, 2), cross(2, 0), cross(0, 1)))

    def forced(self, n, amp=None):
        m = self.m
        on = (m.kx == 0) & (m.kz == 0) & (m.ky == self.kw["kf"])
        return torch.cat([n[:2], (n[2] + (-0.5 * self.kw["kf"]) * on)[None], n[3:]])

    def step3(self, w):
        m, dt, nu = self.m, self.dt, self.kw["v2"] * self.m.k2
        if self.fl == "euler":
            a = self.rhs3(w)
            p = w + dt * a
            return m.L * (p + 0.5 * dt * (self.rhs3(p) - m.L * a))
        n1 = dt / (1 + 0.5 * nu * dt) * m.L
        a = self.forced(self.rhs3(w))
        p = n1 * ((1 - 0.5 * nu * dt) / dt * w + a)
        return m.L * (p + 0.5 * n1 * (self.forced(self.rhs3(p)) - a))

    def rhs4(self, z):
        m, ri = self.m, self.kw["ri"]
        s, co = math.sin(self.kw["theta"]), math.cos(self.kw["theta"])
        out = torch.empty_like(z)
        out[:3] = self.rhs3(z[:3])
        bx, by, bz = (1j * k * z[3] for k in (m.kx, m.ky, m.kz))
        out[0] -= ri * (by * s - bz * co)
        out[1] += ri * bx * s
        out[2] -= ri * bx * co
        u = [a * m.ki for a in m.curl(*m.fill(z[:3]))]
        r = m.fill(z[3:])[0]
        adv = sum(m.grid(a) * m.grid(1j * k * r) for a, k in zip(u, (m.kx, m.ky, m.kz)))
        v = [a * m.ki for a in m.curl(*z[:3])]
        out[3] = v[1] * co + v[2] * s - m.modes(adv)
        return out

    def step4(self, x):
        m, dt, q = self.m, self.dt, self.kw["v2"] * self.m.k2       # Sc = 1: one damping for all fields
        z, acc = x, 0
        for weight, frac, h in ((1 / 6, 0.25, 0.5), (1 / 3, 0.25, 0.5), (1 / 3, 0.5, 1.0)):
            c = self.forced(m.L * self.rhs4(z))
            acc = acc + weight * dt * c
            z = (1 - frac * dt * q) / (1 + frac * dt * q) * (x + h * dt * c)
        c = self.forced(self.rhs4(z))
        half = 0.5 * dt * q
        r = m.L * ((1 - half) * x + acc + dt * c / 6) / (1 + half)
        div = (m.kx * r[0] + m.ky * r[1] + m.kz * r[2]) * m.ki
        for f, k in enumerate((m.kx, m.ky, m.kz)):
            r[f] -= k * div
        return r

    def steps(self, z, n):
        step = {"ns2d": self.step2, "bous": self.step4}.get(self.fl, self.step3)
        for _ in range(n):
            z = step(z[0])[None] if self.fl == "ns2d" else step(z)
        return z


def exact(case, seed):
    c = case
    m = Modes(c)
    f = Flow(c)
    shape = (FIELDS[c["flavour"]],) + m.shape
    if c["kind"] == "tangent":
        z = states(c, seed, 1 + c["extra"])
        f.dt = span(c, f.dt) / c["steps"]
        out = []
        for d in z[1:]:
            a, b = z[0].reshape(m.shape), d.reshape(m.shape)
            for _ in range(c["steps"]):
                a, b = f.step2(a, b)
            out.append(b.reshape(1, -1))
        return {"flow": a.reshape(1, -1), "jv": torch.stack(out)}
    if c["kind"] == "adjoint":
        z, lam = (a.reshape(shape) * m.L for a in states(c, seed, 2))
        traj = [z]
        for _ in range(c["steps"]):
            traj.append(f.step3(traj[-1]))
        for w in traj[-2::-1]:
            w = w.detach().requires_grad_()
            lam, = torch.autograd.grad(f.step3(w), w, lam)
        return {"flow": traj[-1].reshape(3, -1), "gradient": (m.L * lam).reshape(3, -1)}
    z = states(c, seed, c["batch"])
    for i in range(c["batch"]):
        z[i] = f.steps(z[i].reshape(shape), c["steps"]).reshape(z[i].shape)
    out = {"state": z}
    if c["diag"]:
        e = m.L * (z[0].reshape(shape)[:3].abs() ** 2).sum(0)
        shell = (m.k2.sqrt() + 0.5).long()
        spec = torch.zeros(c["ny"] // 3 + 2, dtype=torch.float64, device="cuda")
        keep = shell < spec.numel()
        spec.index_add_(0, shell[keep], (e * m.ki)[keep])
        out.update(energy=float((e * m.ki).sum()), enstrophy=float(e.sum()) * (2 if m.two else 1),
                   spectrum=spec)
    return out
