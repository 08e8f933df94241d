"""The workloads this framework is timed on: what a user has it do, through its public entry points.

Every case starts from the initial condition of decaying isotropic turbulence that the framework's own runs use (solenoidal
velocity with E(k) ~ k^4 exp(-2 (k / k0)^2), uniform density and pressure), drawn here on the GPU from the case's seed.

  step      one Eulerian step on device buffers the caller owns (no allocation, no copy): the smallest call
  run       Context.run: steps with the device's CFL dt, then the state as the caller's array
  dropin    the reference's evolveEulerian: state up, one step, state down
  coupled   the evolve loop with tracers: dt, coupled step, ...; tracers, statistics and (where asked) the state come back
  ensemble  independent runs with tracers stepped together from a captured graph
  gradient  the adjoint gradient of the final kinetic energy
  diagnose  the output phase of a run: flow statistics, samples and all 41 properties at every tracer
"""
import ctypes
import math

import numpy as np
import torch

from dns_gkm_lpt_amd import _lib as gl
from dns_gkm_lpt_amd import adjoint

R_GAS, GAM, RHO0, T0, PRN = 287.0, 1.4, 1.0, 300.0, 0.7
P0 = RHO0 * R_GAS * T0
CFL = 0.5


def listed():
    return [
        # a serving loop or a captured graph that owns its buffers: one step of the smallest production grid
        dict(name="step_32_fp64", kind="step", nc=32, mixed=False, Mt=0.3, Re=30.0),
        # the 32^3 validation run (Mt 0.3, Re_lambda 30), a stretch of it
        dict(name="run_32_fp64", kind="run", nc=32, mixed=False, Mt=0.3, Re=30.0, steps=50),
        # a grid that no tile divides, in the default precision of throughput runs
        dict(name="run_100_mixed", kind="run", nc=100, mixed=True, Mt=0.3, Re=40.0, steps=50),
        # the size of the reference's production run, in the reference's precision
        dict(name="run_256_fp64", kind="run", nc=256, mixed=False, Mt=0.488, Re=100.0, steps=12),
        # the headline grid in mixed precision, up to a field output
        dict(name="run_512_mixed", kind="run", nc=512, mixed=True, Mt=0.5, Re=100.0, steps=10),
        # the drop-in path: a host program that calls the step on its own arrays
        dict(name="dropin_64_fp64", kind="dropin", nc=64, mixed=False, Mt=0.3, Re=40.0),
        # the 128^3 configuration with 2^18 tracers (Mt 0.3, Re_lambda 50), a stretch of it
        dict(name="coupled_128_fp64", kind="coupled", nc=128, mixed=False, Mt=0.3, Re=50.0, tracers=1 << 18, steps=25, state=True),
        # the headline grid with 2^22 tracers: a stretch between two tracer outputs
        dict(name="coupled_512_mixed", kind="coupled", nc=512, mixed=True, Mt=0.5, Re=100.0, tracers=1 << 22, steps=5, state=False),
        # a parameter study: members of the three grid sizes of the ensemble configuration
        dict(name="ensemble_20_mixed", kind="ensemble", n32=8, n48=8, n64=4, mixed=True, tracers=8192, steps=50),
        # gradient of the 64^3 problem (Mt 0.3, Re_lambda 40) over a shorter horizon, checkpointed
        dict(name="gradient_64", kind="gradient", nc=64, Mt=0.3, Re=40.0, steps=10, every=4),
        # an output step of the 128^3 configuration: statistics line, tracer samples and tracer properties
        dict(name="diagnose_128", kind="diagnose", nc=128, mixed=False, Mt=0.3, Re=50.0, tracers=1 << 18),
        # an output step of a larger mixed run, few tracers
        dict(name="diagnose_240_mixed", kind="diagnose", nc=240, mixed=True, Mt=0.4, Re=60.0, tracers=100_003),
    ]


def draw(rng):
    def size(lo, hi):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return min(hi, max(lo, n - n % 8 if rng.random() < 0.5 and n - n % 8 >= lo else n))

    flow = dict(Mt=round(rng.uniform(0.1, 0.6), 3), Re=round(rng.uniform(20.0, 100.0), 1))
    mixed = rng.random() < 0.5
    kind = rng.choice(["step", "run", "run", "dropin", "coupled", "coupled", "ensemble", "gradient", "diagnose"])
    if kind == "step":
        return dict(kind=kind, nc=size(16, 64), mixed=mixed, **flow)
    if kind == "run":
        nc = size(24, 288)
        return dict(kind=kind, nc=nc, mixed=mixed, steps=max(2, min(60, int(2e8 / nc ** 3))), **flow)
    if kind == "dropin":
        return dict(kind=kind, nc=size(32, 160), mixed=mixed, **flow)
    if kind == "coupled":
        nc = size(32, 224)
        np_ = int(math.exp(rng.uniform(math.log(1 << 10), math.log(1 << 20))))
        return dict(kind=kind, nc=nc, mixed=mixed, tracers=np_, steps=max(2, min(30, int(6e7 / nc ** 3))),
                    state=rng.random() < 0.7, **flow)
    if kind == "ensemble":
        return dict(kind=kind, n32=rng.randint(1, 8), n48=rng.randint(0, 8), n64=rng.randint(0, 4), mixed=mixed,
                    tracers=rng.choice([1000, 4096, 8192, 10_001]), steps=rng.randint(10, 50))
    if kind == "gradient":
        return dict(kind=kind, nc=size(20, 64), steps=rng.randint(3, 10), every=rng.randint(1, 5), **flow)
    return dict(kind=kind, nc=size(32, 240), mixed=mixed, tracers=int(math.exp(rng.uniform(math.log(1 << 10), math.log(1 << 20)))), **flow)


# ---- inputs -----------------------------------------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _velocity(nc, Mt, seed, k0=4.0, kmax=8):
    """Solenoidal band-limited random velocity (3, nc, nc, nc) over (y, x, z), components (u, v, w) along (x, y, z)."""
    dev = _device()
    g = torch.Generator(device="cpu").manual_seed(int(seed))
    kmax = min(kmax, nc // 2 - 1)
    m = 2 * kmax + 1
    a = torch.randn((3, m, m, kmax + 1, 2), generator=g, dtype=torch.float64)
    k = torch.arange(-kmax, kmax + 1, dtype=torch.float64)
    ky, kx, kz = k[:, None, None], k[None, :, None], k[kmax:][None, None, :]
    k2 = (ky * ky + kx * kx + kz * kz).clamp(min=1e-14)
    kk = k2.sqrt()
    amp = torch.where((kk >= 1) & (kk <= kmax), kk * torch.exp(-((kk / k0) ** 2)), torch.zeros_like(kk))
    c = torch.view_as_complex(a)
    dot = (kx * c[0] + ky * c[1] + kz * c[2]) / k2
    c = torch.stack([c[0] - dot * kx, c[1] - dot * ky, c[2] - dot * kz]) * amp
    full = torch.zeros((3, nc, nc, nc // 2 + 1), dtype=torch.complex128, device=dev)
    at = (torch.arange(-kmax, kmax + 1) % nc).to(dev)
    full[:, at[:, None], at[None, :], : kmax + 1] = c.to(dev)
    u = torch.stack([torch.fft.irfftn(full[q], s=(nc, nc, nc)) for q in range(3)])
    del full
    return u * (Mt * math.sqrt(GAM * P0 / RHO0) / (u * u).sum(0).mean().sqrt())


def _params(u, Mt, Re):
    """The record of gas and flow parameters a run is configured with; viscosity from Re_lambda."""
    dx = 2 * math.pi / u.shape[-1]
    ek = 0.5 * float((u * u).sum(0).mean())
    sq = 0.0
    for q in range(3):
        for ax in range(3):
            sq += float(((0.5 / dx) * (torch.roll(u[q], -1, ax) - torch.roll(u[q], 1, ax))).square().mean())
    return dict(gam=GAM, rho0=RHO0, Mt=float(Mt), Re=float(Re), mu0=2 * ek * math.sqrt(5 / (3 * sq)) / Re, p0=P0,
                t0=math.sqrt(10 * ek / sq) / math.sqrt(2 * ek / 3))


def _conserved(u):
    """(5, nc, nc, nc) conserved variables of velocity u with uniform density and pressure."""
    W = torch.empty((5,) + u.shape[1:], dtype=torch.float64, device=u.device)
    W[0] = RHO0
    W[1:4] = RHO0 * u
    W[4] = RHO0 * (P0 / (RHO0 * (GAM - 1.0)) + 0.5 * (u * u).sum(0))
    return W


def _padded(W):
    """The host layout: three periodic ghost layers on every face."""
    nc = W.shape[-1]
    at = (torch.arange(-3, nc + 3) % nc).to(W.device)
    return torch.stack([w[at][:, at][:, :, at] for w in W])


def _flow(case, seed, nc=None):
    u = _velocity(nc or case["nc"], case["Mt"], seed)
    return _conserved(u), _params(u, case["Mt"], case["Re"])


def _tracers(n, seed):
    g = torch.Generator(device="cpu").manual_seed(int(seed) + 1_000_003)
    return torch.rand((n, 3), generator=g, dtype=torch.float64) * (2 * math.pi)


def _context(case, W, P):
    c = gl.Context(W.shape[-1], P, cfl=CFL, precision=gl.GKM_MIXED if case["mixed"] else gl.GKM_FP64)
    c.upload(_padded(W).cpu().numpy())
    return c


def _members(case, seed):
    """[(nc, Mt, Re, seed of the member)] of an ensemble case: each member its own flow."""
    out = []
    for nc, n in ((32, case["n32"]), (48, case["n48"]), (64, case["n64"])):
        for _ in range(n):
            m = len(out)
            r = np.random.default_rng([int(seed), m])
            out.append((nc, float(r.uniform(0.1, 0.6)), float(r.uniform(20, 60)), 1000 * int(seed) + m))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        ms = _members(case, seed)
        flows = []
        for nc, Mt, Re, s in ms:
            u = _velocity(nc, Mt, s)
            flows.append((_conserved(u), _params(u, Mt, Re)))
        ens = gl.Ensemble([m[0] for m in ms], [P for _, P in flows], cfl=CFL,
                          precision=gl.GKM_MIXED if case["mixed"] else gl.GKM_FP64)
        for c, (W, _), m in zip(ens.members, flows, ms):
            c.upload(_padded(W).cpu().numpy())
            c.lpt_upload(_tracers(case["tracers"], m[3]).numpy())
        return dict(case=case, ens=ens)
    if kind == "gradient":
        u = _velocity(case["nc"], case["Mt"], seed)
        P = _params(u, case["Mt"], case["Re"])
        dt = float(_cfl_dt(_conserved(u)[:, None])[0])
        pb = adjoint.Problem(case["nc"], P, dt, case["steps"], case["every"])
        return dict(case=case, problem=pb, u=u.cpu().numpy())
    W, P = _flow(case, seed)
    if kind == "step":
        cfg = gl.make_config(case["nc"], P, CFL, gl.GKM_MIXED if case["mixed"] else gl.GKM_FP64)
        return dict(case=case, cfg=cfg, W=W, out=torch.empty_like(W), dt=float(_cfl_dt(W[:, None])[0]),
                    msg=ctypes.create_string_buffer(256))
    if kind == "dropin":
        c = gl.Context(case["nc"], P, cfl=CFL, precision=gl.GKM_MIXED if case["mixed"] else gl.GKM_FP64)
        return dict(case=case, ctx=c, W=_padded(W).cpu().numpy(), dt=float(_cfl_dt(W[:, None])[0]))
    c = _context(case, W, P)
    if kind == "diagnose":
        c.run(SPUN_UP)
    if kind in ("coupled", "diagnose"):
        c.lpt_upload(_tracers(case["tracers"], seed).numpy())
    return dict(case=case, ctx=c)


SPUN_UP = 3  # steps before the output of a diagnose case: density and pressure are no longer uniform
STATS = ("tke", "diss", "sijsij", "prms", "trms", "vrms", "pmean", "tmean", "vmean", "enstrophy")


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "step":
        rc = gl.lib().gkm_step_noalloc(ctypes.byref(state["cfg"]), state["W"].data_ptr(), state["out"].data_ptr(), state["dt"],
                                       torch.cuda.current_stream().cuda_stream, state["msg"], 256)
        if rc:
            raise RuntimeError(state["msg"].value.decode())
        return state["out"]
    if kind == "run":
        dts = state["ctx"].run(case["steps"], record_dt=True)
        return dict(dt=dts, W=state["ctx"].download())
    if kind == "dropin":
        c = state["ctx"]
        c.upload(state["W"])
        c.step(state["dt"])
        return c.download()
    if kind == "coupled":
        c = state["ctx"]
        dts = []
        for _ in range(case["steps"]):
            dts.append(c.cfl_dt())
            c.lpt_coupled_step(dts[-1])
        pos, vel = c.lpt_download()
        out = dict(dt=np.array(dts), pos=pos, vel=vel)
        if case["state"]:
            out["W"] = c.download()
        return out
    if kind == "ensemble":
        ens = state["ens"]
        ens.run(case["steps"], graph=True)
        out = dict(dt=ens.dt())
        for m, c in enumerate(ens.members):
            pos, vel = c.lpt_download()
            out["m%02d" % m] = dict(W=c.download(), pos=pos, vel=vel)
        return out
    if kind == "gradient":
        J, g = state["problem"].gradient(state["u"])
        return dict(J=J, g=g)
    c = state["ctx"]
    s = c.stats()
    U, gU, gV, gW = c.lpt_sample()
    p = c.lpt_stats()
    flow = [getattr(s, k) for k in STATS] + list(s.skew) + list(s.kurt)
    return dict(flow=np.array(flow), tracer=np.array([p.tke, p.sijsij, p.skew_u, p.skew_w]), U=U, gU=gU, gV=gV, gW=gW,
                props=c.lpt_properties())


def work(case):
    """Per cell and step: the state read once and written once, and about 3700 operations a face (both WENO sides of five
    variables and the gas-kinetic flux in its reduced form), three faces a cell.  Per spline: 24 bytes a knot.  Per tracer:
    its positions, velocities and 64 coefficients a field, which neighbouring tracers share (one read of the field)."""
    kind = case["kind"]
    if kind == "ensemble":
        cells = case["n32"] * 32 ** 3 + case["n48"] * 48 ** 3 + case["n64"] * 64 ** 3
        np_ = case["tracers"] * (case["n32"] + case["n48"] + case["n64"])
    else:
        cells, np_ = case["nc"] ** 3, case.get("tracers", 0)
    steps = case.get("steps", 1)
    state = 40.0 * cells
    step = dict(bytes=2 * state, flops=11100.0 * cells)
    spline = dict(bytes=state + 48.0 * cells, flops=3 * 30.0 * cells)
    tracer = dict(bytes=24.0 * cells + 144.0 * np_, flops=2 * 3 * 300.0 * np_)
    if kind in ("step", "run"):
        return dict(bytes=steps * step["bytes"] + (state if kind == "run" else 0), flops=steps * step["flops"])
    if kind == "dropin":
        return dict(bytes=2 * step["bytes"], flops=step["flops"])
    if kind in ("coupled", "ensemble"):
        per = {k: step[k] + spline[k] + tracer[k] for k in step}
        return dict(bytes=steps * per["bytes"] + 48.0 * np_ + (state if case.get("state", True) else 0), flops=steps * per["flops"])
    if kind == "gradient":
        # forward, one recomputation of all but the last segment, and a reverse pass of about three forward ones
        again = max(0, steps - case["every"])
        return dict(bytes=(4 * steps + again) * step["bytes"], flops=(4 * steps + again) * step["flops"])
    return dict(bytes=3 * state + 8 * 16.0 * cells + np_ * 8.0 * (3 + 12 + 41), flops=11 * 30.0 * cells + 100.0 * cells + 5000.0 * np_)


# ---- the same in 64 bits with plain torch -------------------------------------------------------------------------------
# States are (5, B, n, n, n) over (variable, member, y, x, z), unpadded and periodic.

def _col(v, W):
    return torch.as_tensor(v, dtype=torch.float64, device=W.device).reshape(-1, 1, 1, 1)


def _cfl_dt(W):
    d = W[0]
    V2 = (W[1] ** 2 + W[2] ** 2 + W[3] ** 2) / d ** 2
    p = d * (GAM - 1) * (W[4] / d - 0.5 * V2)
    top = (V2.sqrt() + (GAM * p / d).sqrt()).flatten(1).amax(1)
    return CFL * (2 * math.pi / W.shape[-1]) / top


def _pressure(W):
    return (GAM - 1) * (W[4] - 0.5 * (W[1] ** 2 + W[2] ** 2 + W[3] ** 2) / W[0])


def _weno(a, b, c, d, e, f):
    """Six cells around a face -> the value at the face from the left (WENO-SYMOO)."""
    q0 = (2 * a - 7 * b + 11 * c) / 6
    q1 = (-b + 5 * c + 2 * d) / 6
    q2 = (2 * c + 5 * d - e) / 6
    q3 = (11 * d - 7 * e + 2 * f) / 6
    s0 = 13 / 12 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2
    s1 = 13 / 12 * (b - 2 * c + d) ** 2 + 0.25 * (d - b) ** 2
    s2 = 13 / 12 * (c - 2 * d + e) ** 2 + 0.25 * (-3 * c + 4 * d - e) ** 2
    s3 = 13 / 12 * (d - 2 * e + f) ** 2 + 0.25 * (-5 * d + 8 * e - 3 * f) ** 2
    s3 = torch.maximum(torch.maximum(s0, s1), torch.maximum(s2, s3))
    w = [g / (1e-10 + s) for g, s in ((0.05, s0), (0.45, s1), (0.45, s2), (0.05, s3))]
    return (w[0] * q0 + w[1] * q1 + w[2] * q2 + w[3] * q3) / (w[0] + w[1] + w[2] + w[3])


K_INT = int((5.0 - 3.0 * GAM) / (GAM - 1.0))


class _Gas:
    """A Maxwellian in the frame that moves with its tangential velocity; `tab` is its table of normal moments."""

    def __init__(self, W):
        self.d, self.u, self.v, self.w = W[0], W[1] / W[0], W[2] / W[0], W[3] / W[0]
        self.lam = 0.5 * self.d / _pressure(W)
        self.th = 0.5 / self.lam

    def full(self):
        t = [torch.ones_like(self.u), self.u]
        for i in range(2, 7):
            t.append(self.u * t[-1] + (i - 1) * self.th * t[-2])
        return t

    def half(self, sign):
        """Moments over sign * u > 0."""
        s = self.lam.sqrt()
        t = [0.5 * torch.erfc(-sign * s * self.u)]
        t.append(self.u * t[0] + sign * 0.5 * torch.exp(-self.lam * self.u ** 2) / (math.sqrt(math.pi) * s))
        for i in range(2, 7):
            t.append(self.u * t[-1] + (i - 1) * self.th * t[-2])
        return t

    def into(self, m):
        """Lab frame -> this state's tangential frame."""
        return [m[0], m[1], m[2] - self.v * m[0], m[3] - self.w * m[0],
                m[4] - self.v * m[2] - self.w * m[3] + 0.5 * (self.v ** 2 + self.w ** 2) * m[0]]

    def back(self, m):
        return [m[0], m[1], m[2] + self.v * m[0], m[3] + self.w * m[0],
                m[4] + self.v * m[2] + self.w * m[3] + 0.5 * (self.v ** 2 + self.w ** 2) * m[0]]

    def slope(self, b):
        """Micro slope of a macro slope b (this frame), with the Prandtl number on the energy part."""
        q = self.u ** 2 + (K_INT + 3) * self.th
        r2 = b[1] - self.u * b[0]
        a4 = (2 * b[4] - b[0] * q - 2 * self.u * r2) * (4 * self.lam ** 2) / ((K_INT + 3) * PRN)
        a1 = 2 * self.lam * r2 - self.u * a4
        return [b[0] - a1 * self.u - 0.5 * a4 * q, a1, 2 * self.lam * b[2], 2 * self.lam * b[3], a4]

    def mom(self, t, k):
        """<u^k psi> in this frame; psi = (1, u, v, w, energy)."""
        z = torch.zeros_like(t[k])
        return [t[k], t[k + 1], z, z, 0.5 * (t[k + 2] + (K_INT + 2) * self.th * t[k])]

    def moma(self, t, k, a, c=0):
        """<u^k psi (a . psi)>; c = 2 or 3: with the tangential velocity v or w of this frame in the weight too."""
        th, K2, K4 = self.th, K_INT + 2, K_INT + 4
        h0, h1, h2 = t[k], t[k + 1], t[k + 2]
        if c == 0:
            s1, s2 = 0.5 * (h2 + K2 * th * h0), 0.5 * (t[k + 3] + K2 * th * h1)
            s4 = 0.25 * (t[k + 4] + 2 * K2 * th * h2 + K2 * K4 * th * th * h0)
            return [a[0] * h0 + a[1] * h1 + a[4] * s1, a[0] * h1 + a[1] * h2 + a[4] * s2, a[2] * th * h0, a[3] * th * h0,
                    a[0] * s1 + a[1] * s2 + a[4] * s4]
        s = 0.5 * th * (h2 + K4 * th * h0)
        m = [a[c] * th * h0, a[c] * th * h1, 0.0, 0.0, a[c] * s]
        m[c] = a[0] * th * h0 + a[1] * th * h1 + a[4] * s
        return m

    def flux3(self, t, k, ax, ay, az):
        """<u^k (u ax + V ay + W az) . psi psi> with V, W the lab-frame tangential velocities, seen in this frame."""
        vw = [self.v * y + self.w * z for y, z in zip(ay, az)]
        return _add(self.moma(t, k + 1, ax), self.moma(t, k, ay, 2), self.moma(t, k, az, 3), self.moma(t, k, vw))


def _add(*ms):
    return [sum(c[1:], c[0]) for c in zip(*ms)]


def _times(s, m):
    return [s * x for x in m]


def _face_flux(WL, WR, Wl, Wr, D, tau, dt, dx):
    """Time-integrated gas-kinetic flux of a face; D: slopes (x left, x right, y left, ...), all in the face's frame."""
    L, R = _Gas(Wl), _Gas(Wr)
    hl, hr = L.half(1.0), R.half(-1.0)
    We = _add(L.back(_times(L.d, L.mom(hl, 0))), R.back(_times(R.d, R.mom(hr, 0))))
    E = _Gas(We)
    ep, en, ef = E.half(1.0), E.half(-1.0), E.full()
    pl, pr = L.d / L.lam, R.d / R.lam
    tau = tau + dt * (pl - pr).abs() / (pl + pr).abs()
    ex = torch.exp(-dt / tau)
    g0 = dt - tau * (1 - ex)
    g1 = -(1 - ex) / g0
    g2 = (-dt + 2 * tau * (1 - ex) - dt * ex) / g0
    g4 = (dt * ex - tau * (1 - ex)) / g0
    g5 = -tau * g1
    P = tau * (1 - ex)
    Q = -tau * dt * ex + tau * tau * (1 - ex)
    p0 = dt - P
    p1, p2, p4, p5 = 0.5 * dt * dt - tau * p0, Q - tau * p0, -Q - tau * P, -tau * P
    Be = [0.0] * 5
    F = _times(p0 * E.d, E.back(E.mom(ef, 1)))
    bye, bze = [0.0] * 5, [0.0] * 5
    for side, (S, h) in enumerate(((L, hl), (R, hr))):
        ax, ay, az = (S.slope(S.into(_times(1 / S.d, D[2 * d + side]))) for d in range(3))
        A = S.slope(_times(-1.0, S.flux3(S.full(), 0, ax, ay, az)))
        bye = _add(bye, S.back(S.moma(h, 0, ay)))
        bze = _add(bze, S.back(S.moma(h, 0, az)))
        Be = _add(Be, S.back(_times(S.d, _add(_times(g4 + g5, S.flux3(h, 0, ax, ay, az)), _times(g5, S.moma(h, 0, A))))))
        F = _add(F, S.back(_times(S.d, _add(_times(P, S.mom(h, 1)), _times(p4, S.flux3(h, 1, ax, ay, az)), _times(p5, S.moma(h, 1, A))))))
    s = 2.0 / (E.d * dx)
    al = E.slope(E.into([(We[q] - WL[q]) * s for q in range(5)]))
    ar = E.slope(E.into([(WR[q] - We[q]) * s for q in range(5)]))
    ay, az = E.slope(E.into(bye)), E.slope(E.into(bze))
    vw = [E.v * y + E.w * z for y, z in zip(ay, az)]

    def both(k):
        return _add(E.moma(ep, k + 1, al), E.moma(en, k + 1, ar), E.moma(ef, k, ay, 2), E.moma(ef, k, az, 3), E.moma(ef, k, vw))

    # the zeroth moments of the equilibrium and of the two halves are the same state, with weights that cancel
    Be = _add(Be, E.back(_times(g2 * E.d, both(0))))
    A = E.slope(E.into(_times(1 / E.d, Be)))
    return _add(F, E.back(_times(E.d, _add(_times(p1, E.moma(ef, 1, A)), _times(p2, both(1))))))


def _sweep(W, dt, mu0, axis):
    """Flux differences of one direction; axis 0, 1, 2 = x, y, z."""
    dx = 2 * math.pi / W.shape[-1]
    t0 = P0 / (R_GAS * RHO0)
    dims = {0: 2, 1: 1, 2: 3}  # x, y, z -> dimension of a (B, y, x, z) array
    n = dims[axis] - 4
    # tangential neighbours: (y, z) for x, (x, z) for y, (x, y) for z
    ta, tb = ((dims[1] - 4, -1), (dims[0] - 4, -1), (dims[0] - 4, dims[1] - 4))[axis]
    swap = (1, 2, 3)[axis]
    T = _pressure(W) / (R_GAS * W[0])
    S = torch.cat([W[:4], T[None]])
    s = [torch.roll(S, 2 - i, n) for i in range(6)]

    def state(r):
        out = torch.empty_like(r)
        out[:4] = r[:4]
        out[4] = r[0] * R_GAS * r[4] / (GAM - 1) + 0.5 * (r[1] ** 2 + r[2] ** 2 + r[3] ** 2) / r[0]
        return out if not r.requires_grad else torch.cat([r[:4], (r[0] * R_GAS * r[4] / (GAM - 1) + 0.5 * (r[1] ** 2 + r[2] ** 2 + r[3] ** 2) / r[0])[None]])

    l, r = state(_weno(*s)), state(_weno(*s[::-1]))
    WR = torch.roll(W, -1, n)
    D = [2 * (l - W) / dx, 2 * (WR - r) / dx]
    for d in (ta, tb):
        D += [0.5 * (torch.roll(x, -1, d) - torch.roll(x, 1, d)) / dx for x in (l, r)]
    tau = mu0 * (T / t0) ** 1.5 * (t0 + 110.4) / (T + 110.4) / (R_GAS * W[0] * T)
    turn = [0, swap, 2, 3, 4]
    turn[swap] = 1
    F = _face_flux(*([x[q] for q in turn] for x in (W, WR, l, r)), [[x[q] for q in turn] for x in D], tau, dt, dx)
    F = torch.stack([F[q] for q in turn])
    return F - torch.roll(F, 1, n)


def _exact_step(W, dt, mu0):
    dx = 2 * math.pi / W.shape[-1]
    out = W.clone()
    for axis in range(3):
        out = out - _sweep(W, dt, mu0, axis) / dx
    return out


def _solve(n, device):
    """(n + 2, n): knot values of a line -> coefficients of its natural cubic spline."""
    A = torch.zeros((n + 2, n + 2), dtype=torch.float64)
    i = torch.arange(n)
    A[i + 1, i], A[i + 1, i + 1], A[i + 1, i + 2] = 1 / 6, 4 / 6, 1 / 6
    A[0, :3] = torch.tensor([1.0, -2.0, 1.0], dtype=torch.float64)
    A[-1, -3:] = A[0, :3]
    B = torch.zeros((n + 2, n), dtype=torch.float64)
    B[i + 1, i] = 1.0
    return torch.linalg.solve(A, B).to(device)


def _along(M, f, dim):
    f = f.movedim(dim, 0)
    shape = f.shape
    return (M @ f.reshape(shape[0], -1)).reshape((M.shape[0],) + shape[1:]).movedim(0, dim)


def _coefs(f):
    """Natural tricubic spline of a padded field (nt, nt, nt) over (y, x, z)."""
    M = _solve(f.shape[0], f.device)
    for d in range(3):
        f = _along(M, f, d)
    return f.contiguous()


def _pad3(f):
    at = (torch.arange(-3, f.shape[-1] + 3) % f.shape[-1]).to(f.device)
    return f[at][:, at][:, :, at]


def _weights(t):
    t2, t3 = t * t, t * t * t
    w = torch.stack([(1 - t) ** 3 / 6, (3 * t3 - 6 * t2 + 4) / 6, (-3 * t3 + 3 * t2 + 3 * t + 1) / 6, t3 / 6])
    d = torch.stack([-0.5 * (1 - t) ** 2, 1.5 * t2 - 2 * t, -1.5 * t2 + t + 0.5, 0.5 * t2])
    return w, d, torch.stack([1 - t, 3 * t - 2, 1 - 3 * t, t])


def _evaluate(c, dx, pos, order=1):
    """Value (np,), gradient (np, 3) and Hessian (np, 9) over (y, x, z) of a spline at positions (y, x, z)."""
    n = c.shape[0]
    u = (pos + 2.5 * dx) / dx
    i = u.floor().long()
    ws = [_weights((u - i)[:, a]) for a in range(3)]
    flat = c.reshape(-1)
    sums = {}
    wanted = [(0, 0, 0)]
    if order > 0:
        wanted += [(1, 0, 0), (0, 1, 0), (0, 0, 1)]
    if order > 1:
        wanted += [(2, 0, 0), (1, 1, 0), (1, 0, 1), (0, 2, 0), (0, 1, 1), (0, 0, 2)]
    for a in range(4):
        for b in range(4):
            row = ((i[:, 0] + a) * n + i[:, 1] + b) * n + i[:, 2]
            v = [flat[row + k] for k in range(4)]
            lines = [sum(ws[2][o][k] * v[k] for k in range(4)) for o in range(order + 1)]
            for w in wanted:
                sums[w] = sums.get(w, 0.0) + ws[0][w[0]][a] * ws[1][w[1]][b] * lines[w[2]]
    val = sums[(0, 0, 0)]
    grad = torch.stack([sums[w] for w in wanted[1:4]], 1) / dx if order else None
    hess = None
    if order > 1:
        h = [sums[w] for w in wanted[4:]]
        hess = torch.stack([h[0], h[1], h[2], h[1], h[3], h[4], h[2], h[4], h[5]], 1) / dx ** 2
    return val, grad, hess


def _velocity_splines(W):
    return [_coefs(_pad3(W[q] / W[0])) for q in (1, 2, 3)]


def _sample(cs, dx, pos):
    return torch.stack([_evaluate(c, dx, pos, 0)[0] for c in cs], 1)


def _heun(cs, dx, pos, U, dt):
    """U = (u, v, w) at the start, positions (y, x, z); the predictor is not wrapped, the result is."""
    turn = [1, 0, 2]
    U2 = _sample(cs, dx, pos + dt * U[:, turn])
    return torch.remainder(pos + 0.5 * dt * (U + U2)[:, turn], 2 * math.pi)


def _most(case):
    """Whether the plain version takes a few seconds and not many."""
    if case["kind"] == "ensemble":
        return True
    n = case["nc"] ** 3
    if case["kind"] == "gradient":
        return case["nc"] <= 64
    return n * case.get("steps", 1) <= 2.5e8


def _exact_coupled(W, pos, mu0, steps):
    """Members of one size: W (5, B, ...), pos: a list of positions.  Returns W, pos, velocities at the last step, dts."""
    dx = 2 * math.pi / W.shape[-1]
    cs = [_velocity_splines(W[:, m]) for m in range(W.shape[1])] if pos else None
    dts, U = [], None
    for _ in range(steps):
        dt = _cfl_dt(W)
        dts.append(dt)
        W1 = _exact_step(W, dt.reshape(-1, 1, 1, 1), mu0)
        if pos:
            U = [_sample(c, dx, x) for c, x in zip(cs, pos)]
            cs = [_velocity_splines(W1[:, m]) for m in range(W.shape[1])]
            pos = [_heun(c, dx, x, v, float(t)) for c, x, v, t in zip(cs, pos, U, dt)]
        W = W1
    return W, pos, U, torch.stack(dts)


def _gradients_at_knots(c, dx):
    w, d = (torch.tensor(v, dtype=torch.float64) for v in ((1 / 6, 4 / 6, 1 / 6), (-0.5, 0.0, 0.5)))

    def line(f, v, dim):
        n = f.shape[dim] - 2
        return sum(float(v[k]) * f.narrow(dim, k, n) for k in range(3))

    return [line(line(line(c, d if a == 0 else w, 0), d if a == 1 else w, 1), d if a == 2 else w, 2) / dx for a in range(3)]


def _exact_diagnose(W, P, pos):
    nc = W.shape[-1]
    dx = 2 * math.pi / nc
    t0 = P0 / (R_GAS * RHO0)
    cs = _velocity_splines(W)
    inner = (slice(3, -3),) * 3
    g = [[x[inner] for x in _gradients_at_knots(c, dx)] for c in cs]  # g[component][y, x, z]
    p = _pressure(W)
    T, vol = p / (R_GAS * W[0]), 1 / W[0]
    mu = P["mu0"] * (T / t0) ** 1.5 * (t0 + 110.4) / (T + 110.4)
    ux, uy, uz = g[0][1], g[0][0], g[0][2]
    vx, vy, vz = g[1][1], g[1][0], g[1][2]
    wx, wy, wz = g[2][1], g[2][0], g[2][2]

    def sij(ux, uy, uz, vx, vy, vz, wx, wy, wz):
        return ux ** 2 + vy ** 2 + wz ** 2 + 0.5 * ((uy + vx) ** 2 + (uz + wx) ** 2 + (wy + vz) ** 2)

    def shape(x, k):
        return float((x ** k).mean() / (x ** 2).mean() ** (k / 2))

    mt2 = P["Mt"] ** 2
    flow = [(W[1:4] ** 2).sum(0).div(W[0]).mean(), (mu * sum(x * x for r in g for x in r)).mean(), sij(ux, uy, uz, vx, vy, vz, wx, wy, wz).mean(),
            (p - p.mean()).square().mean().sqrt() / (GAM * P["p0"] * mt2), (T - T.mean()).square().mean().sqrt() / ((GAM - 1) * t0 * mt2),
            (vol - vol.mean()).square().mean().sqrt() / (mt2 / P["rho0"]), p.mean(), T.mean(), vol.mean(),
            ((wy - vz) ** 2 + (uz - wx) ** 2 + (vx - uy) ** 2).mean()]
    flow = [float(x) for x in flow] + [shape(x, 3) for x in (ux, vy, wz)] + [shape(x, 4) for x in (ux, vy, wz)]
    del g, mu, T, vol
    at = [_evaluate(c, dx, pos) for c in cs]
    U = torch.stack([a[0] for a in at], 1)
    gU, gV, gW = (a[1] for a in at)
    tr = [float((U * U).sum(1).mean()),
          float(sij(gU[:, 1], gU[:, 0], gU[:, 2], gV[:, 1], gV[:, 0], gV[:, 2], gW[:, 1], gW[:, 0], gW[:, 2]).mean()),
          shape(gU[:, 1], 3), shape(gW[:, 2], 3)]
    d, pp = _evaluate(_coefs(_pad3(W[0])), dx, pos), _evaluate(_coefs(_pad3(p)), dx, pos, 2)
    lap = []
    for c in cs:
        k, w = (torch.tensor(v, dtype=torch.float64, device=c.device) for v in ((1.0, -2.0, 1.0), (1 / 6, 4 / 6, 1 / 6)))
        f = 0.0
        for a in range(3):
            t = c
            for b in range(3):
                n = t.shape[b] - 2
                t = sum(float((k if a == b else w)[j]) * t.narrow(b, j, n) for j in range(3))
            f = f + t
        lap.append(_evaluate(_coefs(f / dx ** 2), dx, pos))
    props = torch.cat([d[0][:, None], U, pp[0][:, None], d[1], gU, gV, gW, pp[1], torch.stack([x[0] for x in lap], 1), pp[2]] + [x[1] for x in lap], 1)
    return dict(flow=np.array(flow), tracer=np.array(tr), U=U, gU=gU, gV=gV, gW=gW, props=props)


def _exact_gradient(u, P, dt, steps):
    from torch.utils.checkpoint import checkpoint

    u = u.clone().requires_grad_(True)
    W = torch.cat([torch.full_like(u[:1], RHO0), RHO0 * u, (P0 / (GAM - 1) + 0.5 * RHO0 * (u * u).sum(0))[None]])[:, None]
    dt, mu0, dx = _col(dt, u), _col(P["mu0"], u), 2 * math.pi / u.shape[-1]
    for _ in range(steps):
        W = W - sum(checkpoint(_sweep, W, dt, mu0, axis, use_reentrant=False) for axis in range(3)) / dx
    J = (0.5 * (W[1] ** 2 + W[2] ** 2 + W[3] ** 2) / W[0]).mean()
    J.backward()
    return dict(J=float(J.detach()), g=u.grad)


def exact(case, seed):
    if not _most(case):
        return None
    kind = case["kind"]
    dev = _device()
    if kind == "ensemble":
        ms = _members(case, seed)
        out, dts = {}, [0.0] * len(ms)
        for nc in (32, 48, 64):
            at = [m for m in range(len(ms)) if ms[m][0] == nc]
            if not at:
                continue
            us = [_velocity(nc, ms[m][1], ms[m][3]) for m in at]
            mu0 = _col([_params(u, ms[m][1], ms[m][2])["mu0"] for u, m in zip(us, at)], us[0])
            W = torch.stack([_conserved(u) for u in us], 1)
            W, pos, U, dt = _exact_coupled(W, [_tracers(case["tracers"], ms[m][3]).to(dev) for m in at], mu0, case["steps"])
            for i, m in enumerate(at):
                out["m%02d" % m] = dict(W=_padded(W[:, i]), pos=pos[i], vel=U[i])
                dts[m] = float(dt[-1, i])
        return dict(dt=np.array(dts), **out)
    if kind == "gradient":
        u = _velocity(case["nc"], case["Mt"], seed)
        return _exact_gradient(u, _params(u, case["Mt"], case["Re"]), float(_cfl_dt(_conserved(u)[:, None])[0]), case["steps"])
    W, P = _flow(case, seed)
    mu0 = _col(P["mu0"], W)
    if kind == "diagnose":
        W = _exact_coupled(W[:, None], [], mu0, SPUN_UP)[0][:, 0]
        return _exact_diagnose(W, P, _tracers(case["tracers"], seed).to(dev))
    if kind in ("step", "dropin"):
        W = _exact_step(W[:, None], _cfl_dt(W[:, None]).reshape(-1, 1, 1, 1), mu0)[:, 0]
        return W if kind == "step" else _padded(W)
    pos = [_tracers(case["tracers"], seed).to(dev)] if kind == "coupled" else []
    W, pos, U, dt = _exact_coupled(W[:, None], pos, mu0, case["steps"])
    if kind == "run":
        return dict(dt=dt[:, 0], W=_padded(W[:, 0]))
    out = dict(dt=dt[:, 0], pos=pos[0], vel=U[0])
    if case["state"]:
        out["W"] = _padded(W[:, 0])
    return out
