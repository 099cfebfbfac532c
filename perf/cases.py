"""The work a program has this framework do, as cases that can be timed and compared.

One pass is what a host program does per output interval: `calls` AlgoGas
calls of length DT (twenty per orbit at r = 1) through the public entry
points, the torque log after each where one is kept, and the state copied to
host arrays at the end.  The state carries on from pass to pass, as in a run.

listed()             the cases
draw(rng)            one more of the same ranges
prepare(case, seed)  inputs from the seed, and the disc / batch / network that a program keeps
run(state)           one pass and its outputs
work(case)           bytes and operations one pass cannot do without
exact(case, seed)    what run() returns the first time, in 64 bits by plain torch / numpy

Storage: `fp` 64 or 32 is the disc's field type.  Fields of a disc with FP32
storage are handed on as float32 (they hold no more).  The two velocity
components are handed on as one array: the radial one is a small part of a
flow that rotates, and its rounding is set by the other.
"""
import math

import numpy as np
import torch

from dustyfargoadsg_amd import _capi
from dustyfargoadsg_amd.disc import Batch, Disc, init_dust_system, make_planets
from dustyfargoadsg_amd.surrogate import MLP
from dustyfargoadsg_amd.workloads import SIGMA0_ST1_CM, batch_discs, default_params, gas_dust, gas_dust_particles

DT = 2 * math.pi / 20
NO_PLANETS = dict(dist=[], mass=[], acc=[], feel_disk=[], feel_others=[])


def listed():
    return [
        # the discs the warm start's network is trained on, one by itself: six or so
        # sub-steps of six short kernels in each call
        gas("planet_64x192_f32", 64, 192, 32, 20, planet="fixed"),
        # the shape of the quick-start parameter file (200 x 400, isothermal, alpha
        # 1e-4), its planet free to migrate, the torque logged after every call; rings
        # that are no multiple of a wavefront
        gas("template_200x400_f64", 200, 400, 64, 20, planet="free", alpha=1e-4, viscosity=0.0, log=True),
        # locally isothermal disc with a planet on a fixed orbit, the plain method in FP64
        gas("planet_128x384_f64", 128, 384, 64, 20, planet="fixed", log=True),
        # a C host that keeps the fields itself: arrays in and out on every call,
        # with the energy equation
        gas("energy_256x768_f64_host", 256, 768, 64, 5, energy=True, alpha=1e-3, viscosity=0.0, host=True),
        # adiabatic, self-gravitating, beta-cooled disc: the benchmark's disc, both storage types
        gas("energy_sg_512x1536_f32", 512, 1536, 32, 5, energy=True, sg=True, alpha=1e-3, viscosity=0.0),
        gas("energy_sg_512x1536_f64", 512, 1536, 64, 5, energy=True, sg=True, alpha=1e-3, viscosity=0.0),
        # the largest grid: gas, self-gravity and a planet in FP32; gas and a planet in FP64
        gas("gas_sg_1024x3072_f32", 1024, 3072, 32, 3, sg=True, planet="fixed", alpha=1e-3, viscosity=0.0),
        gas("planet_1024x3072_f64", 1024, 3072, 64, 3, planet="fixed", alpha=1e-3, viscosity=0.0),
        # 10^6 grains of 1 mm - 1 cm in the largest gas disc, CIC, drag feedback
        dict(name="dust_1024x3072_f32", kind="dust", nrad=1024, nsec=3072, fp=32, calls=3, particles=1_000_000,
             interp=1, feedback=True),
        # the second fluid with its momentum equations and diffusion, a ragged grid
        dict(name="dust_fluid_150x450_f64", kind="fluid", nrad=150, nsec=450, fp=64, calls=5, sfta=False,
             diffusion=True, feedback=True),
        # a parameter sweep: uneven discs advanced together
        dict(name="sweep_16_discs_f32", kind="batch", discs=16, nrads="64 128 256", fp=32, calls=5),
        # training the warm start's network on a sweep's profiles
        dict(name="mlp_train_2048", kind="mlp", batch=2048, steps=20),
    ]


def gas(name, nrad, nsec, fp, calls, *, energy=False, sg=False, planet="none", alpha=0.0, viscosity=1e-5, log=False,
        host=False):
    c = dict(kind="gas", nrad=nrad, nsec=nsec, fp=fp, calls=calls, energy=energy, sg=sg, planet=planet, alpha=alpha,
             viscosity=viscosity, log=log, host=host)
    return dict(c, name=name) if name else c


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _ring(rng, nrad):
    """A ring of two to four times as many cells as there are rings, of any size the grid takes."""
    ns = int(nrad * rng.uniform(2.0, 4.0))
    step = 1 if ns <= 1024 else 2 if ns <= 1536 else 4 if ns <= 2048 else 12
    return min(ns - ns % step, 3072)


def _alpha(rng):
    return float("%.2e" % 10 ** rng.uniform(-4.0, -2.3))


def _calls(nrad):
    """Calls between two outputs: an orbit of a small disc, fewer of a large one."""
    return 20 if nrad <= 150 else 5 if nrad <= 400 else 3


def draw(rng):
    kind = rng.choice(["gas", "gas", "gas", "sg", "sg", "dust", "fluid", "batch", "mlp"])
    fp = rng.choice([32, 64])
    if kind == "gas":
        nrad = _log_uniform(rng, 48, 900)
        energy = rng.random() < 0.4
        alpha = rng.choice([0.0, _alpha(rng)])
        planet = "none" if energy else rng.choice(["none", "fixed", "free"])
        return gas(None, nrad, _ring(rng, nrad), fp, _calls(nrad), energy=energy, planet=planet, alpha=alpha,
                   viscosity=0.0 if alpha else 1e-5, log=fp == 64 and planet != "none" and rng.random() < 0.5,
                   host=nrad <= 400 and rng.random() < 0.25)
    if kind == "sg":
        nrad = rng.choice([64, 128, 256, 512])
        nsec = rng.choice([2, 3, 4]) * nrad
        energy = rng.random() < 0.6
        return gas(None, nrad, nsec, fp, _calls(nrad), energy=energy, sg=True, planet="none" if energy else "fixed",
                   alpha=_alpha(rng), viscosity=0.0)
    if kind == "dust":
        nrad = _log_uniform(rng, 64, 500)
        return dict(kind="dust", nrad=nrad, nsec=_ring(rng, nrad), fp=fp, calls=3,
                    particles=_log_uniform(rng, 10_000, 500_000), interp=rng.choice([0, 1, 2]),
                    feedback=rng.random() < 0.7)
    if kind == "fluid":
        nrad = _log_uniform(rng, 64, 400)
        return dict(kind="fluid", nrad=nrad, nsec=_ring(rng, nrad), fp=64, calls=_calls(nrad), sfta=rng.random() < 0.5,
                    diffusion=rng.random() < 0.5, feedback=rng.random() < 0.5)
    if kind == "batch":
        nrads = "%d %d" % (_log_uniform(rng, 48, 128), _log_uniform(rng, 64, 256))
        return dict(kind="batch", discs=rng.randint(3, 16), nrads=nrads, fp=fp, calls=5)
    return dict(kind="mlp", batch=rng.randint(65, 2048), steps=rng.randint(5, 20))


# ---------------------------------------------------------------------------
# inputs

def _params(case):
    """The disc of a case and its planet (the columns of a planet file)."""
    k = case["kind"]
    if k == "dust":
        return gas_dust(case["nrad"], case["nsec"], add_noise=0)
    free = case.get("planet") == "free"
    p = default_params(
        nrad=case["nrad"], nsec=case["nsec"], rmin=0.4, rmax=2.5, log_grid=1, sigma0=6.3662e-4, sigma_slope=0.5,
        aspect_ratio=0.05, flaring_index=0.0, viscosity=case.get("viscosity", 1e-5),
        alpha_viscosity=case.get("alpha", 0.0), thickness_smoothing=0.6, forced_circular=0 if free else 1,
        boundary=_capi.BC_WALL, fast_transport=1)
    if case.get("energy"):
        # Sigma ~ 1/r with the smallest Toomre Q at 2, beta cooling
        p.rmax, p.sigma_slope = 4.0, 1.0
        p.sigma0 = 0.05 / (math.pi * 2.0 * 4.0)
        p.energy_equation, p.beta_cooling, p.beta_cooling_time, p.viscous_heating = 1, 1, 10.0, 1
    if k == "fluid":
        # 1 cm grains have Stokes numbers near 0.2 at r = 1
        p.sigma0 = 5 * SIGMA0_ST1_CM
    if case.get("sg"):
        p.self_gravity, p.sg_thickness_smoothing = 1, 0.3
    if k == "gas" and case["planet"] == "none":
        return p, NO_PLANETS
    f = int(free)
    return p, dict(dist=[1.0], mass=[3e-4 if free else 1e-3], acc=[0.0], feel_disk=[f], feel_others=[0])


def _noise(p, seed):
    """The start's relative density noise, 1e-3, ring nrad empty."""
    g = torch.Generator().manual_seed(seed)
    return 1.0 + 1e-3 * (2.0 * torch.rand(p.nrad, p.nsec, generator=g, dtype=torch.float64).numpy() - 1.0)


def _rmed(p):
    edge = p.rmin * np.exp(np.arange(p.nrad + 1) / p.nrad * math.log(p.rmax / p.rmin))
    ri, rs = edge[:-1], edge[1:]
    return edge, 2.0 / 3.0 * (rs ** 3 - ri ** 3) / (rs ** 2 - ri ** 2)


def _density(p, seed):
    rho = np.zeros((p.nrad + 1, p.nsec))
    rho[:-1] = (p.sigma0 * _rmed(p)[1] ** -p.sigma_slope)[:, None] * _noise(p, seed)
    return rho


def _energy(p):
    r = _rmed(p)[1]
    e = np.zeros((p.nrad + 1, p.nsec))
    e[:-1] = (p.sigma0 * r ** -p.sigma_slope * p.aspect_ratio ** 2 * r ** (2 * p.flaring_index - 1.0) /
              (p.adiabatic_index - 1.0))[:, None]
    return e


def _disc(p, planets, fp, seed, fluid=None):
    d = Disc(p, _capi.FP64 if fp == 64 else _capi.FP32)
    if fluid is not None:
        d.attach_dust_fluid(fluid)
    rho = _density(p, seed).ravel()
    en = _energy(p).ravel() if p.energy_equation else None
    sys_ = make_planets(p, planets)
    vr, vt = d.init_euler(rho, en, sys_)
    return d, dict(rho=rho, vr=vr, vt=vt, energy=en, planets=sys_)


def _batch_params(case, seed):
    """Planet mass, viscosity, aspect ratio, flaring and slope of each disc from the seed; the sizes in turn."""
    sizes = [int(x) for x in case["nrads"].split()]
    got = batch_discs(case["discs"], seed, nrads=sizes[:1])
    for k, (p, _) in enumerate(got):
        p.nrad, p.add_noise = sizes[k % len(sizes)], 0
        p.nsec = 3 * p.nrad
    return got


def _profiles(case, seed):
    """Features in [-1, 1] and gap-like profiles on 256 radii, as the network is trained on."""
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, (case["batch"], 4)).astype(np.float32)
    r = np.linspace(0.4, 2.5, 256)
    t = 1.0 - (0.5 + 0.4 * x[:, :1]) * np.exp(-((r - 1.0) / (0.15 + 0.05 * x[:, 1:2])) ** 2) + 0.1 * x[:, 2:3] * (r - 1.45)
    w = []
    for n_in, n_out in zip([4, 256, 256, 256], [256] * 4):
        lim = math.sqrt(6.0 / (n_in + n_out))
        w += [rng.uniform(-lim, lim, n_in * n_out), np.zeros(n_out)]
    return x, t.astype(np.float32), np.concatenate(w).astype(np.float32)


def prepare(case, seed):
    s = dict(case=case)
    if case["kind"] == "mlp":
        s["x"], s["t"], w = _profiles(case, seed)
        s["net"] = MLP(max_batch=2048, seed=1)
        s["net"].set_params(w)
        return s
    if case["kind"] == "batch":
        s["discs"] = [_disc(p, pl, case["fp"], seed + k)[0] for k, (p, pl) in enumerate(_batch_params(case, seed))]
        s["batch"] = Batch(s["discs"])
        return s
    p, planets = _params(case)
    fluid = None
    if case["kind"] == "fluid":
        fluid = _capi.dust_fluid_default_params(sfta=int(case["sfta"]), sizepart=1e-3 if case["sfta"] else 1e-2,
                                                rhopart=2.7, dust_diffusion=int(case["diffusion"]),
                                                dust_feedback=int(case["feedback"]))
    s["disc"], s["st"] = _disc(p, planets, case["fp"], seed, fluid)
    if case["kind"] == "dust":
        # with feedback the shortest stopping time limits the time step: no grains below 1 mm
        dp = gas_dust_particles(p, case["particles"], seed=seed, interpolation=case["interp"],
                                dust_feedback=int(case["feedback"]), sizeminpart=1e-3 if case["feedback"] else 1e-6)
        s["disc"].attach_dust(dp, init_dust_system(p, dp), DT)
    return s


# ---------------------------------------------------------------------------
# one pass

def _fields(st, fp, energy):
    t = np.float32 if fp == 32 else np.float64
    v = np.empty((2, st["vr"].size), t)
    v[0], v[1] = st["vr"], st["vt"]
    out = dict(rho=st["rho"].astype(t, copy=False), velocity=v)
    if energy:
        out["energy"] = st["energy"].astype(t, copy=False)
    return out


def _planets(sys_):
    n = sys_.nb
    return np.array([list(a)[:n] for a in (sys_.x, sys_.y, sys_.vx, sys_.vy)])


def run(s):
    case = s["case"]
    if case["kind"] == "mlp":
        loss = s["net"].train(s["x"], s["t"], case["steps"])
        return dict(loss=np.float32(loss), weights=s["net"].params())
    if case["kind"] == "batch":
        for _ in range(case["calls"]):
            s["batch"].algogas(DT)
        return [_fields(d.state(), case["fp"], False) for d in s["discs"]]
    d, st, log = s["disc"], s["st"] if case.get("host") else None, []
    for _ in range(case["calls"]):
        d.algogas(DT, st)
        if case.get("log"):
            log.append(d.update_log())
    if st is None:
        st = d.state()
    out = _fields(st, case["fp"], case.get("energy"))
    if log:
        out["torque"], out["indirect"] = np.stack([a for a, _ in log]), np.stack([b for _, b in log])
    if case.get("planet", "none") != "none":
        out["planets"] = _planets(st["planets"])
    if case["kind"] == "fluid":
        f = d.dust_fluid()
        out["dust_rho"], out["stokes"] = f["drho"], f["stokes"]
        out["dust_velocity"] = np.stack([f["dvr"], f["dvt"]])
    if case["kind"] == "dust":
        q = d.dust_state()
        t = np.float32 if case["fp"] == 32 else np.float64
        out["position"] = np.stack([q["r"], q["th"]]).astype(t, copy=False)
        out["particle_velocity"] = np.stack([q["vr"], q["vth"]]).astype(t, copy=False)
        out["stokes"] = q["stokesnb"].astype(t, copy=False)
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _substeps(p):
    """The sub-steps of one call by the CFL condition on the smooth initial disc
    (sound speed, viscosity, shear)."""
    edge, r = _rmed(p)
    dx = np.minimum(edge[1:] - edge[:-1], r * 2 * math.pi / p.nsec)
    cs = p.aspect_ratio * r ** (p.flaring_index - 0.5)
    nu = p.alpha_viscosity * cs ** 2 * r ** 1.5 if p.alpha_viscosity else p.viscosity + 0.0 * r
    if p.energy_equation:
        cs = cs * math.sqrt(p.adiabatic_index)
    dt = np.min(0.5 / np.hypot(cs / dx, 4.0 * nu / dx ** 2))
    om = r ** -1.5
    dt = min(dt, np.min(math.pi / p.nsec / np.abs(om[1:] - om[:-1])))
    return math.ceil(DT / dt)


def _gas_work(p, fp, calls):
    """Per sub-step: every state field read and written once, with self-gravity the
    two kernel spectra read; the state to the host once.  Operations: the stencils'
    (source terms, viscosity, six quantities in three transport passes, CFL) and the
    transforms' (5 n log2 n)."""
    w, cells, n = fp // 8, p.nrad * p.nsec, calls * _substeps(p)
    ns = 3 + bool(p.energy_equation)
    bytes_ = n * cells * w * (2 * ns + (4 if p.self_gravity else 0)) + cells * w * ns
    flops = 600.0 + (150.0 if p.energy_equation else 0.0)
    if p.self_gravity:
        flops += 2 * 5 * math.log2(p.nsec) + 4 * 5 * math.log2(2 * p.nrad) + 30
    return bytes_, n * cells * flops, n


def work(case):
    if case["kind"] == "mlp":
        n = 4 * 256 + 3 * 256 * 256
        b, k = case["batch"], case["steps"]
        act = b * 2 * (4 + 3 * 256) + b * 4 * 256
        return dict(bytes=float(k * (n * 4 * 8 + 2 * act)), flops=float(k * 6 * b * n))
    if case["kind"] == "batch":
        got = [_gas_work(p, case["fp"], case["calls"]) for p, _ in _batch_params(case, 1)]
        return dict(bytes=float(sum(b for b, _, _ in got)), flops=float(sum(f for _, f, _ in got)))
    p, _ = _params(case)
    b, f, n = _gas_work(p, case["fp"], case["calls"])
    if case["kind"] == "dust":
        # per particle five values in and four out; the feedback grids
        b += n * (72 * case["particles"] + (4 * case["fp"] // 8 * p.nrad * p.nsec if case["feedback"] else 0))
        f += n * 400.0 * case["particles"]
    if case["kind"] == "fluid":
        b, f = 2 * b, 2 * f
    return dict(bytes=float(b), flops=float(f))


# ---------------------------------------------------------------------------
# the same in 64 bits, whole arrays at a time

def exact(case, seed):
    if case["kind"] == "mlp":
        return _mlp_exact(case, seed)
    if case["kind"] == "batch":
        out = []
        for k, (p, planets) in enumerate(_batch_params(case, seed)):
            out.append(_gas_exact(p, planets, seed + k, case["calls"], False))
        return out
    if case["kind"] != "gas":
        return None
    p, planets = _params(case)
    return _gas_exact(p, planets, seed, case["calls"], case["log"])


def _mlp_exact(case, seed):
    """Full-batch Adam on a GELU network, mean squared error."""
    x, t, flat = _profiles(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x, t, flat = (torch.from_numpy(a).to(dev, torch.float64) for a in (x, t, flat))
    w, off = [], 0
    for n_in in (4, 256, 256, 256):
        w.append(flat[off:off + n_in * 256].reshape(n_in, 256).clone().requires_grad_())
        w.append(flat[off + n_in * 256:off + (n_in + 1) * 256].clone().requires_grad_())
        off += (n_in + 1) * 256

    def loss():
        h = x
        for k in range(0, 8, 2):
            h = h @ w[k] + w[k + 1]
            if k < 6:
                h = torch.nn.functional.gelu(h)
        return ((h - t) ** 2).mean()

    opt = torch.optim.Adam(w, lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
    for _ in range(case["steps"]):
        opt.zero_grad()
        loss().backward()
        opt.step()
    with torch.no_grad():
        return dict(loss=loss().cpu().numpy()[()], weights=torch.cat([a.detach().ravel() for a in w]).cpu().numpy())


class _Grid:
    """Ring tables as (nrad, 1) columns, azimuths as a row."""

    def __init__(self, p, dev):
        edge, r = _rmed(p)
        col = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)[:, None]
        self.nr, self.ns, self.dphi = p.nrad, p.nsec, 2 * math.pi / p.nsec
        self.edge, self.r_np = edge, r
        self.rinf, self.rsup, self.r = col(edge[:-1]), col(edge[1:]), col(r)
        self.dr = self.rsup - self.rinf
        self.drm = torch.ones_like(self.r)
        self.drm[1:] = self.r[1:] - self.r[:-1]
        self.surf = math.pi * (self.rsup ** 2 - self.rinf ** 2) / p.nsec
        phi = self.dphi * torch.arange(p.nsec, device=dev, dtype=torch.float64)[None, :]
        self.x, self.y = self.r * torch.cos(phi), self.r * torch.sin(phi)
        self.dx = self.r * self.dphi
        self.sigma = col(p.sigma0 * r ** -p.sigma_slope)
        self.e_floor = 1e-3 * self.sigma * p.aspect_ratio ** 2 * self.r ** (2 * p.flaring_index - 1) / (p.adiabatic_index - 1)
        self.cs = col(p.aspect_ratio * r ** (p.flaring_index - 0.5))


def _prev(a):
    return torch.roll(a, 1, 1)


def _next(a):
    return torch.roll(a, -1, 1)


def _below(a):
    """The ring below each ring (ring 0: itself)."""
    return torch.cat([a[:1], a[:-1]])


def _gravity(p, g, dev):
    """Accelerations of a density by the zero-padded convolution in log r and phi."""
    nr, ns = g.nr, g.ns
    eps, rstep = p.sg_thickness_smoothing * p.aspect_ratio, math.log(p.rmax / p.rmin) / nr
    u = np.log(g.edge / g.edge[0])
    u = torch.from_numpy(np.concatenate([u[:nr], -u[nr:0:-1]])).to(dev)[:, None]
    phi = g.dphi * torch.arange(ns, device=dev, dtype=torch.float64)[None, :]
    den = (eps * eps * torch.exp(u) + 2.0 * (torch.cosh(u) - torch.cos(phi))) ** -1.5
    kr = torch.fft.rfft2((1.0 + eps * eps - torch.cos(phi) * torch.exp(-u)) * den)
    kt = torch.fft.rfft2(torch.sin(phi) * den)
    q = g.r / g.r[0]

    def accel(rho):
        pad = rho.new_zeros(2 * nr, ns)
        pad[:nr] = rho * torch.sqrt(q)
        ar = torch.fft.irfft2(torch.fft.rfft2(pad) * kr, s=(2 * nr, ns))[:nr]
        pad[:nr] = rho * q ** 1.5
        at = torch.fft.irfft2(torch.fft.rfft2(pad) * kt, s=(2 * nr, ns))[:nr]
        c = rstep * g.dphi
        return -c * ar / torch.sqrt(q) + rho * c / eps, -c * at / q ** 1.5

    return accel


def _rk5(q, dt, m):
    """Cash-Karp step of one body around the star (indirect term of its own mass)."""
    def f(v):
        d3 = math.hypot(v[0], v[1]) ** 3
        return dt * np.array([v[2], v[3], -(1.0 + m) * v[0] / d3, -(1.0 + m) * v[1] / d3])
    a = [[], [0.2], [0.075, 0.225], [0.3, -0.9, 1.2], [-11 / 54, 2.5, -70 / 27, 35 / 27],
         [1631 / 55296, 175 / 512, 575 / 13824, 44275 / 110592, 253 / 4096]]
    k = []
    for row in a:
        k.append(f(q + sum((c * ki for c, ki in zip(row, k)), np.zeros(4))))
    return q + 37 / 378 * k[0] + 250 / 621 * k[2] + 125 / 594 * k[3] + 512 / 1771 * k[5]


def _stress(g, rho, vr, vt, nu):
    """div v and the viscous stresses; vr holds nrad + 1 faces."""
    lo, hi = vr[:-1], vr[1:]
    dvt = (_next(vt) - vt) / g.dx
    div = (hi * g.rsup - lo * g.rinf) / g.dr / g.r + dvt
    trr = 2 * rho * nu * ((hi - lo) / g.dr - div / 3)
    tpp = 2 * rho * nu * (dvt + 0.5 * (hi + lo) / g.r - div / 3)
    drp = 0.5 * (g.rinf * (vt / g.r - _below(vt / g.r)) / g.drm + (lo - _prev(lo)) / (g.dphi * g.rinf))
    trp = 0.5 * (rho + _below(rho) + _prev(rho) + _prev(_below(rho))) * nu * drp
    trp[0] = 0
    return div, trr, tpp, trp


def _limited(dm, dp):
    """dm dp / (dm + dp) where both have one sign, else 0."""
    q = dm * dp
    return torch.where(q > 0, q / torch.where(q > 0, dm + dp, torch.ones_like(q)), torch.zeros_like(q))


def _radial_star(g, w, v, dt):
    """Upwind value at faces 1 .. nrad-1 (v: the velocity there)."""
    d = (w[1:] - w[:-1]) / g.drm[1:]
    s = torch.zeros_like(w)
    s[1:-1] = 2 * _limited(d[:-1], d[1:])
    up = torch.zeros_like(w)
    up[:-1] = g.drm[1:]  # distance to the next ring; the last ring has no slope
    return torch.where(v > 0, w[:-1] + 0.5 * (up[:-1] - v * dt) * s[:-1], w[1:] - 0.5 * (up[1:] + v * dt) * s[1:])


def _azimuthal_pass(g, q, v, dt):
    def star(w):
        s = _limited(w - _prev(w), _next(w) - w) / g.dx
        return torch.where(v * dt > 0, _prev(w) + (g.dx - v * dt) * _prev(s), w - (g.dx + v * dt) * s)
    rho = q[-1]
    rs = star(rho) * v * (g.dr * dt / g.surf)
    out = []
    for a in q:
        f = star(a / (rho + 1e-20)) * rs
        out.append(a + f - _next(f))
    return out


def _gas_exact(p, planets, seed, calls, log):
    """AlgoGas calls of length DT from the initial state, and the torque log."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = _Grid(p, dev)
    nr, ns, energy, gam = g.nr, g.ns, bool(p.energy_equation), p.adiabatic_index
    rho = torch.from_numpy(_density(p, seed)).to(dev)[:nr]
    en = torch.from_numpy(_energy(p)).to(dev)[:nr] if energy else None
    accel = _gravity(p, g, dev) if p.self_gravity else None

    def sound():
        return torch.sqrt(gam * (gam - 1.0) * en / rho) if energy else g.cs.expand(nr, ns)

    def viscosity(cs):
        if p.alpha_viscosity:
            return p.alpha_viscosity * cs.mean(1, keepdim=True) ** 2 * g.r ** 1.5
        return p.viscosity * torch.ones_like(g.r)

    cs = sound()
    nu = viscosity(cs)
    # initial velocities: rotation against pressure and the disc's own gravity, viscous drift
    f, sl = p.flaring_index, p.sigma_slope
    vt2 = (1.0 - p.aspect_ratio ** 2 * g.r ** (2 * f) * (1 + sl - 2 * f)) / g.r
    m = float(np.float32(planets["mass"][0])) if planets["dist"] else 0.0
    pl = np.array([1.0, 0.0, -1e-10 * math.sqrt(1 + m), math.sqrt(1 + m)]) if m else None
    if accel:
        axi = accel(rho)[0].mean(1, keepdim=True)
        vt2 = vt2 - g.r * axi
        if m:
            k = min(int(np.searchsorted(g.r_np, 1.0, side="right")), nr - 2)
            ri, rj, a = g.r_np[k], g.r_np[k + 1], axi[:, 0].cpu().numpy()
            pl[3] *= math.sqrt(1.0 - ((1.0 - ri) * a[k + 1] + (rj - 1.0) * a[k]) / (rj - ri) / (1.0 + m))
    vt = torch.sqrt(vt2).expand(nr, ns).clone()
    vt_edge = vt[:, :1].clone()
    vr = torch.zeros(nr + 1, ns, device=dev, dtype=torch.float64)
    vr[:nr] = -3.0 * nu / g.r * ((1.0 - sl + 2 * f) if p.alpha_viscosity else (0.5 - sl))
    smooth = lambda r: p.thickness_smoothing * p.aspect_ratio * r ** (1.0 + f)

    def pull(x, y, soft, cut=None, rings=slice(None)):
        """The disc's pull on a point."""
        dx, dy = g.x - x, g.y - y
        d2 = dx * dx + dy * dy
        a = g.surf * rho / (d2 + soft * soft) ** 1.5
        if cut is not None:
            a = a * cut(torch.sqrt(d2))
        return float((a * dx)[rings].sum()), float((a * dy)[rings].sum())

    done, call, star, logged = 0.0, 0, (0.0, 0.0), []
    while call < calls:
        if done == 0.0:
            cs = sound()
        # time step
        vm = vt.mean(1, keepdim=True)
        lo, hi = vr[:-1], vr[1:]
        small = torch.minimum(g.dr, g.dx)
        dvr, dvt = (hi - lo).neg().clamp_min(0) / g.dr, (_next(vt) - vt).neg().clamp_min(0) / g.dx
        inv2 = ((cs / small) ** 2 + (lo / g.dr) ** 2 + ((vt - vm) / g.dx) ** 2 +
                (4 * 1.41 ** 2 * torch.maximum(dvr, dvt)) ** 2 + (4 * nu / small ** 2) ** 2)
        step = float(0.5 / torch.sqrt(inv2[1:].max()))
        om = vm / g.r
        step = min(step, float((math.pi / ns / (om[:-1] - om[1:]).abs()).min()), DT - done)
        dt = (DT - done) / math.ceil((DT - done) / step)
        done += dt
        cs = sound()
        nu = viscosity(cs)
        # potential: star, planet with its indirect term, the disc's pull on the star
        star = pull(0.0, 0.0, 0.0)
        pot = -1.0 / g.r + star[0] * g.x + star[1] * g.y
        if m:
            d2 = (g.x - pl[0]) ** 2 + (g.y - pl[1]) ** 2
            rp = math.hypot(pl[0], pl[1])
            kick = pull(pl[0], pl[1], smooth(rp)) if planets["feel_disk"][0] else None
            pot = pot - m / torch.sqrt(d2 + smooth(rp) ** 2) + m / rp ** 3 * (g.x * pl[0] + g.y * pl[1])
        if accel:
            sgr, sgt = accel(rho)
        # source terms
        press = (gam - 1.0) * en if energy else rho * cs * cs
        mean_r = 0.5 * (rho + _below(rho))
        vmid = 0.25 * (vt + _next(vt) + _below(vt + _next(vt)))
        acc = -(press - _below(press)) / mean_r / g.drm - (pot - _below(pot)) / g.drm + vmid * vmid / g.rinf
        act = -(press - _prev(press)) / (0.5 * (rho + _prev(rho))) / g.dx - (pot - _prev(pot)) / g.dx
        if accel:
            below = torch.cat([g.r[:1], g.r[:-1]])
            acc = acc + ((g.rinf - below) * sgr + (g.r - g.rinf) * _below(sgr)) / g.drm
            act = act + 0.5 * (sgt + _prev(sgt))
        u = torch.zeros_like(vr)
        u[1:nr] = vr[1:nr] + dt * acc[1:]
        w = vt + dt * act
        # viscosity
        _, trr, tpp, trp = _stress(g, rho, u, w, nu)
        up = torch.cat([trp[1:], trp[:1]])
        fw = ((g.rsup * up - g.rinf * trp) / g.dr + (tpp - _prev(tpp)) / g.dphi + 0.5 * (trp + up)) / g.r
        fu = ((g.r * trr - _below(g.r * trr)) / g.drm + (_next(trp) - trp) / g.dphi - 0.5 * (tpp + _below(tpp))) / g.rinf
        w[1:nr - 1] += (dt * fw / (0.5 * (rho + _prev(rho))))[1:nr - 1]
        u[1:nr] += (dt * fu / mean_r)[1:]
        # artificial viscosity
        du, dw = u[1:] - u[:-1], _next(w) - w
        qr, qt = 1.41 ** 2 * rho * du.clamp_max(0) ** 2, 1.41 ** 2 * rho * dw.clamp_max(0) ** 2
        if energy:
            e = en - dt * (qr * du / g.dr + qt * dw / g.dx)
        u[1:nr] -= (dt * (qr - _below(qr)) / mean_r / g.drm)[1:]
        w = w - dt * (qt - _prev(qt)) / (0.5 * (rho + _prev(rho))) / g.dx
        # heating, compression, cooling
        if energy:
            div, trr, tpp, trp = _stress(g, rho, u, w, nu)
            heat = 0.5 / nu / rho * (trr ** 2 + 2 * trp ** 2 + tpp ** 2) + 2 / 9 * nu * rho * div ** 2
            power = math.log(g.r_np[0] / g.r_np[1]) / math.log(g.r_np[1] / g.r_np[2])
            heat[0] = heat[1] * (heat[1] / heat[2]) ** power
            en = (e + dt * heat) / (1 + (gam - 1.0) * dt * div)
            en = en / (1 + dt * w.mean(1, keepdim=True) / g.r / p.beta_cooling_time)
        # transport: radial, then azimuthal by the residual, the constant residual, the shift
        q = [rho * u[1:], rho * u[:-1], rho * _next(w) * g.r, rho * w * g.r] + ([en] if energy else []) + [rho]
        face = u[1:nr]
        rs = _radial_star(g, rho, face, dt) * face * (dt * g.dphi * g.rinf[1:])
        moved = []
        for a in q:
            flux = torch.zeros_like(u)
            flux[1:nr] = _radial_star(g, a / (rho + 1e-20), face, dt) * rs
            moved.append(a + (flux[:-1] - flux[1:]) / g.surf)
        wm = w.mean(1, keepdim=True)
        turn = wm / g.r * dt / g.dphi
        cells = torch.floor(turn + 0.5)
        moved = _azimuthal_pass(g, moved, w - wm, dt)
        moved = _azimuthal_pass(g, moved, ((turn - cells) * g.dx / dt).expand(nr, ns), dt)
        src = (torch.arange(ns, device=dev)[None, :] - cells.long()) % ns
        moved = [torch.gather(a, 1, src) for a in moved]
        # velocities, floors, walls
        rho = moved[-1]
        vr = torch.zeros_like(u)
        vr[1:nr] = ((_below(moved[0]) + moved[1]) / (rho + _below(rho) + 1e-20))[1:]
        vt = (_prev(moved[2]) + moved[3]) / (rho + _prev(rho) + 1e-20) / g.r
        rho = rho.clamp_min(p.density_floor)
        if energy:
            en = torch.maximum(moved[4], g.e_floor)
        vr[0], vr[nr] = -vr[2], -vr[nr - 2]
        vr[1], vr[nr - 1] = 0, 0
        for i in (0, 1, nr - 2, nr - 1):
            rho[i] = g.sigma[i]
        vt[0], vt[nr - 1] = vt_edge[0], vt_edge[nr - 1]
        # the planet, kicked by the disc as the sub-step found it
        if m:
            if planets["feel_disk"][0]:
                pl[2:] += dt * (np.array(kick) - np.array(star))
            pl = _turn(pl, dt) if p.forced_circular else _rk5(pl, dt, m)
        if done >= 0.999999999 * DT:
            done, call = 0.0, call + 1
            if log:
                # torque and power on the planet: inner and outer disc, whole and without its Hill sphere
                x, y, vx, vy = pl
                r = math.hypot(x, y)
                hill, k = (m / 3.0) ** (1.0 / 3.0) * r, int((g.r_np < r).sum())
                cut = lambda d: torch.sin((d / hill - 0.5).clamp(0.0, 0.5) * math.pi) ** 2
                fs = [pull(x, y, smooth(r), c, part) for c in (None, cut) for part in (slice(0, k), slice(k, nr))]
                logged.append(([[x * b - y * a for a, b in fs] + [vx * a + vy * b for a, b in fs]],
                               [-x * star[1] + y * star[0]]))
    flat = lambda a: torch.cat([a, a.new_zeros(nr + 1 - a.shape[0], ns)]).reshape(-1).cpu().numpy()
    out = dict(rho=flat(rho), velocity=np.stack([flat(vr), flat(vt)]))
    if energy:
        out["energy"] = flat(en)
    if m:
        out["planets"] = pl[:, None]
    if log:
        out["torque"], out["indirect"] = np.array([a for a, _ in logged]), np.array([b for _, b in logged])
    return out


def _turn(pl, dt):
    """A body on a fixed circular orbit."""
    x, y, vx, vy = pl
    r, v = math.hypot(x, y), math.hypot(vx, vy)
    t = math.atan2(y, x) + (x * vy - y * vx) / r ** 2 * dt
    return np.array([r * math.cos(t), r * math.sin(t), -v * math.sin(t), v * math.cos(t)])
