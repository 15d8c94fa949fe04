"""Performance cases: the work users of this framework have it do.

Three paths, all through public entry points:

  rhs    one right-hand side of a state on the device into a device array
         (cns_rhs_noalloc, then cns_sync): a program with its own time
         integrator; its grids end at 2^21 FP64 points.
  run    the reference's main loop body: nsteps steps with the per-step
         statistics, then the state copied to the host arrays the program
         keeps (runSimulation + copyField(1); channels also take the
         wall-normal profiles, as calcAvgChan does).
  batch  many flows advanced together (ensembles, one tick of the serving
         loop), then every member's state.

Arrays are indexed [z, y, x], x unit-stride.  Programs with FP32 storage
keep FP32 fields and records, so theirs are handed over as float32.
"""
import math
from functools import lru_cache

import numpy as np
import torch

import cudanavierstokes_amd as cns


def _case(path, kind, size, order, **kw):
    c = dict(path=path, kind=kind, mx=size[0], my=size[1], mz=size[2], order=order, visc=order, scheme="rk3",
             fp32=False, steps=1)
    c.update(kw)
    return c


def listed():
    cube = lambda n: (n, n, n)  # noqa: E731
    return [
        # smallest calls, latency counts: a right-hand side of the smoke test's box
        dict(_case("rhs", "box", cube(24), 6), name="rhs_box24_o6"),
        # odd sizes, walls on a stretched grid, viscous order below the advective one
        dict(_case("rhs", "channel", (101, 67, 83), 8, visc=4), name="rhs_channel_ragged_o8"),
        # the largest box of the call
        dict(_case("rhs", "box", cube(128), 8), name="rhs_box128_o8"),
        # the reference's default box and scheme: small grid, many steps
        dict(_case("run", "box", cube(64), 4, steps=100), name="run_box64_o4"),
        # the headline benchmark: Taylor-Green 256^3, order 8, classic RK4
        dict(_case("run", "box", cube(256), 8, scheme="rk4", steps=40), name="run_box256_o8_rk4"),
        # the same with FP32 storage
        dict(_case("run", "box", cube(256), 8, scheme="rk4", steps=40, fp32=True), name="run_box256_o8_rk4_fp32"),
        # the reference's channel, both precisions
        dict(_case("run", "channel", (160, 128, 192), 6, steps=50), name="run_channel_o6"),
        dict(_case("run", "channel", (160, 128, 192), 6, steps=50, fp32=True), name="run_channel_o6_fp32"),
        # ragged channel with the reference's other scheme and a lower viscous order
        dict(_case("run", "channel", (90, 75, 110), 6, visc=4, scheme="kutta_rk3", steps=30),
             name="run_channel_ragged_kutta"),
        # the reference's default case, the spatially developing boundary layer
        dict(_case("run", "layer", (240, 64, 2048), 6, visc=4, steps=8), name="run_layer_o6"),
        # an ensemble of independent boxes of the benchmark's sizes (FP32, RK4)
        dict(_case("batch", "boxes", cube(128), 6, scheme="rk4", fp32=True, steps=60, members=12, smallest=32),
             name="batch_ensemble_o6"),
        # one tick of the serving loop: boxes and channels mixed (FP32, RK3)
        dict(_case("batch", "mixed", cube(160), 6, fp32=True, steps=40, members=10, smallest=48),
             name="batch_serving_o6"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    path = rng.choice(["rhs", "run", "run", "run", "batch"])
    order = rng.choice([2, 4, 6, 6, 8, 8])
    visc = order if rng.random() < 0.6 else 2 * rng.randint(1, order // 2)
    if path == "rhs":
        while True:
            s = (size(16, 192), size(16, 192), size(16, 192))
            if s[0] * s[1] * s[2] <= 1 << 21:
                return _case("rhs", rng.choice(["box", "channel"]), s, order, visc=visc)
    scheme = rng.choice(["rk3", "rk3", "kutta_rk3", "rk4"])
    if path == "run":
        kind = rng.choice(["box", "box", "channel", "channel", "layer"])
        if kind == "layer":
            s = (16 * rng.randint(3, 15), size(16, 64), size(160, 1024))
            fp32 = False
        else:
            s = (size(24, 256), size(24, 256), size(24, 256))
            fp32 = rng.random() < 0.4
        most = 40.0 * 256 ** 3 / (s[0] * s[1] * s[2])
        return _case("run", kind, s, order, visc=visc, scheme=scheme, fp32=fp32,
                     steps=max(1, min(rng.randint(8, 100), int(most / 4))))
    kind = rng.choice(["boxes", "mixed"])
    most = size(48, 144)
    return _case("batch", kind, (most, most, most), rng.choice([4, 6, 8]), scheme="rk4" if kind == "boxes" else "rk3",
                 fp32=rng.random() < 0.7, steps=rng.randint(4, 16), members=rng.randint(2, 12), smallest=24)


# ---------------------------------------------------------------------------
# configurations, grids and initial states
# ---------------------------------------------------------------------------

def _config(c):
    kw = dict(scheme=c["scheme"], precision=1 if c["fp32"] else 0, stencil_visc=c["visc"] // 2)
    if c["kind"] == "box":
        return cns.taylor_green(n=c["mx"], order=c["order"], scheme=c["scheme"], Ma=c.get("Ma", 0.1),
                                Re=c.get("Re", 1600.0)).replace(my=c["my"], mz=c["mz"], **kw)
    if c["kind"] == "channel":
        return cns.channel(mx=c["mx"], my=c["my"], mz=c["mz"], order=c["order"], scheme=c["scheme"],
                           Ma=c.get("Ma", 1.5), Re=c.get("Re", 3000.0)).replace(**kw)
    return cns.boundary_layer(mx=c["mx"], my=c["my"], mz=c["mz"], order=c["order"], visc_order=c["visc"],
                              scheme=c["scheme"])


def _members(c, seed):
    """The flows of a batch as single cases, drawn from the seed as the
    ensemble and serving workloads draw theirs."""
    rng = np.random.default_rng([int(seed), 77])
    sizes = [n for n in (32, 48, 64, 96, 128) if n <= c["mx"]] if c["kind"] == "boxes" else None
    out = []
    for k in range(c["members"]):
        ma, re = float(rng.uniform(0.1, 0.4)), float(rng.uniform(400.0, 3000.0))
        # the sizes are the case's, not the seed's: every seed is the same amount of work
        f = 1.0 - k / max(1, c["members"] - 1) * 0.9
        n = int(c["smallest"] + f * (c["mx"] - c["smallest"]))
        if c["kind"] == "boxes":
            n = min(sizes or [n], key=lambda s: abs(s - n)) if c["mx"] == 128 else n
            kind, s = "box", (n, n, n)
        elif k % 3 == 2:
            kind, s, ma = "channel", (n, max(24, 2 * n // 3), max(24, n // 2)), ma + 0.4
        else:
            n = 16 * (n // 16) if n >= 48 else n
            kind, s = "box", (n, n, n)
        out.append(dict(_case("run", kind, s, c["order"], visc=c["visc"], scheme=c["scheme"], fp32=c["fp32"],
                              steps=c["steps"]), Ma=ma, Re=re))
    return out


def _weights(s):
    """central weights: D1 f = sum a_k (f_k - f_-k), D2 f = b_0 f + sum b_k (f_k + f_-k)"""
    f = math.factorial
    a = [0.0] + [(-1) ** (k + 1) * f(s) ** 2 / (k * f(s - k) * f(s + k)) for k in range(1, s + 1)]
    b = [0.0] + [2.0 * a[k] / k for k in range(1, s + 1)]
    b[0] = -2.0 * sum(b[1:])
    return a, b


@lru_cache(maxsize=4)
def _grid(kind, mx, my, mz, s):
    """x, y, z, inverse x metric xp, second metric xpp, cell widths, spacings"""
    g = {}
    box, layer = kind == "box", kind == "layer"
    Lx, Ly, Lz = (2 * math.pi,) * 3 if box else ((20.0, 7.0, 500.0) if layer
                                                 else (2.0, 4 * math.pi / 3, 4 * math.pi))
    dx = Lx / mx
    g["y"], g["z"] = (np.arange(my) + 0.5) * (Ly / my), (np.arange(mz) + 0.5) * (Lz / mz)
    x = (np.arange(mx) + 0.5) * dx
    xp, xpp = np.ones(mx), np.zeros(mx)
    if not box:
        st, den = (5.0, 2.0 * mx) if layer else (1.8, 1.0 * mx)
        t = np.tanh(st * (np.arange(mx + 1) / den - 0.5)) / math.tanh(0.5 * st)
        x = Lx * (1.0 + 0.5 * (t[1:] + t[:-1])) / (1.0 if layer else 2.0)
        a, b = _weights(s)
        e = np.concatenate([-x[:s][::-1], x, 2 * Lx - x[::-1][:s]])
        at = lambda k: e[s + k:s + k + mx]  # noqa: E731
        xp = 1.0 / (sum(a[k] * (at(k) - at(-k)) for k in range(1, s + 1)) / dx)
        xpp = (b[0] * x + sum(b[k] * (at(k) + at(-k)) for k in range(1, s + 1))) / dx / dx
    dxv = np.empty(mx)
    dxv[0], dxv[-1] = (x[1] + x[0]) / 2, Lx - (x[-1] + x[-2]) / 2
    dxv[1:-1] = (x[2:] - x[:-2]) / 2
    g.update(x=x, xp=xp, xpp=xpp, dxv=dxv, dx=dx, dy=Ly / my, dz=Lz / mz, L=(Lx, Ly, Lz))
    return g


def _t(a):
    return torch.as_tensor(a, dtype=torch.float64, device="cuda")


def _layer_reference(c, g, cfg):
    """Laminar profile on [mz][mx] (conserved): Pohlhausen's quartic for the
    streamwise velocity over a layer growing as sqrt(1 + z/Re), temperature
    from the adiabatic Crocco-Busemann relation, uniform pressure."""
    rg = 1.0 / (cfg.gam * cfg.Ma ** 2)
    eta = np.minimum(g["x"][None, :] / np.sqrt(1.0 + g["z"] / cfg.Re)[:, None], 1.0)
    w = 2 * eta - 2 * eta ** 3 + eta ** 4
    r = 1.0 / (1.0 + 0.85 * 0.5 * (cfg.gam - 1) * cfg.Ma ** 2 * (1 - w * w))
    zero = np.zeros_like(r)
    return [r, zero, zero, r * w, rg / (cfg.gam - 1) + 0.5 * r * w * w]


def _layer_sponge(g):
    """strengths of the top, inlet and outlet zones"""
    x, z, (Lx, _, Lz) = g["x"], g["z"], g["L"]
    sx = np.where(x >= Lx - 1.0, (x - (Lx - 1.0)) ** 2, 0.0)
    sz = np.where(z <= 20.0, 0.5 * ((20.0 - z) / 20.0) ** 2, 0.0)
    sz = np.where(z >= Lz - 20.0, 0.5 * ((z - (Lz - 20.0)) / 20.0) ** 2, sz)
    return sx, sz


def _fields(c, seed):
    """rho, u, v, w, rho E [z, y, x] on the GPU: the flow's base state plus
    smooth random velocity and density modes (boxes, layers) or the 10%
    random velocities of the seeded channel."""
    cfg = _config(c)
    g = _grid(c["kind"], c["mx"], c["my"], c["mz"], c["order"] // 2)
    rng = np.random.default_rng([int(seed), 3])
    rg = 1.0 / (cfg.gam * cfg.Ma ** 2)
    Lx, Ly, Lz = g["L"]
    X, Y, Z = _t(g["x"])[None, None, :], _t(g["y"])[None, :, None], _t(g["z"])[:, None, None]
    zero = torch.zeros((c["mz"], c["my"], c["mx"]), dtype=torch.float64, device="cuda")

    def mode(amp):
        f = zero.clone()
        for _ in range(3):
            k, ph, a = rng.integers(1, 4, 3), rng.uniform(0, 2 * math.pi, 3), rng.uniform(-1, 1)
            f += (amp * a * torch.cos(2 * math.pi * int(k[0]) / Lx * X + ph[0]) *
                  torch.cos(2 * math.pi * int(k[1]) / Ly * Y + ph[1]) *
                  torch.cos(2 * math.pi * int(k[2]) / Lz * Z + ph[2]))
        return f

    if c["kind"] == "box":
        x, y, z = 2 * math.pi / Lx * X, 2 * math.pi / Ly * Y, 2 * math.pi / Lz * Z
        u = torch.sin(x) * torch.cos(y) * torch.cos(z) + mode(0.1)
        v = -torch.cos(x) * torch.sin(y) * torch.cos(z) + mode(0.1)
        w = mode(0.1)
        p = rg + (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0) / 16.0
        r = p / rg
    elif c["kind"] == "channel":
        gen = torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + c["mx"])
        noise = lambda: 0.2 * torch.rand(zero.shape, generator=gen, dtype=torch.float64, device="cuda") - 0.1  # noqa
        xi = X / (Lx / 2) - 1.0
        u, v = noise(), noise()
        w = 1.5 * (1.0 - xi * xi) + noise()
        r, p = torch.ones_like(zero), zero + rg
    else:
        ref = [_t(a)[:, None, :] for a in _layer_reference(c, g, cfg)]
        damp = torch.exp(-0.5 * X) * torch.clamp(X, max=1.0)
        r, p = ref[0] + zero, zero + rg
        u, v, w = mode(0.01) * damp, mode(0.01) * damp, ref[3] / ref[0] + mode(0.01) * damp
    return [r, u, v, w, p / (cfg.gam - 1) + 0.5 * r * (u * u + v * v + w * w)]


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

def _solver(c, seed):
    s = cns.Solver(_config(c))
    f = _fields(c, seed)
    if c["kind"] == "layer":
        g = _grid(c["kind"], c["mx"], c["my"], c["mz"], c["order"] // 2)
        s.set_sponge(*_layer_sponge(g), _layer_reference(c, g, s.config))
    s.set_state(*[a.cpu().numpy() for a in f])
    return s, f


def _host(c):
    """the program's own arrays of one state: page-locked, written by every
    copy (and their FP32 twins for FP32 storage)"""
    n = c["mx"] * c["my"] * c["mz"]
    big = [torch.empty(n, dtype=torch.float64, pin_memory=True) for _ in range(5)]
    small = [torch.empty(n, dtype=torch.float32) for _ in range(5)] if c["fp32"] else None
    return big, small


def prepare(case, seed):
    c = dict(case)
    if c["path"] == "batch":
        cs = _members(c, seed)
        solvers = [_solver(m, seed * 131 + k)[0] for k, m in enumerate(cs)]
        return dict(case=c, batch=cns.Batch(solvers), solvers=solvers, host=[_host(m) for m in cs])
    s, f = _solver(c, seed)
    if c["path"] == "rhs":
        r, u, v, w, e = f
        q = torch.stack([r, r * u, r * v, r * w, e]).contiguous()
        return dict(case=c, solver=s, q=q, out=torch.empty_like(q))
    return dict(case=c, solver=s, host=_host(c))


def _state(solver, host):
    big, small = host
    solver._chk(solver.L.cns_get_state(solver.h, *[a.numpy() for a in big]), "cns_get_state")
    if small is None:
        return big
    for a, b in zip(small, big):
        a.copy_(b)
    return small


def run(state):
    c = state["case"]
    if c["path"] == "rhs":
        s = state["solver"]
        s._chk(s.L.cns_rhs_noalloc(s.h, state["q"].data_ptr(), state["out"].data_ptr()), "cns_rhs_noalloc")
        s.sync()
        return state["out"]
    if c["path"] == "batch":
        state["batch"].step(c["steps"])
        return [list(_state(s, h)) for s, h in zip(state["solvers"], state["host"])]
    s = state["solver"]
    kin, enst, time = s.step(c["steps"])
    out = dict(kin=kin, enst=enst, time=time)
    if c["kind"] == "channel":
        out.update(s.channel_profiles())
    if c["fp32"]:
        out = {k: v.astype(np.float32) for k, v in out.items()}
    out["state"] = list(_state(s, state["host"]))
    return out


# ---------------------------------------------------------------------------
# work of one pass
# ---------------------------------------------------------------------------

_WORDS = {"rk3": 50, "kutta_rk3": 65, "rk4": 85}  # words per point and step: stage inputs, operands, outputs
_STAGES = {"rk3": 3, "kutta_rk3": 3, "rk4": 4}


def work(case):
    c = case
    if c["path"] == "batch":
        parts = [work(m) for m in _members(c, 0)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n, s, sv = c["mx"] * c["my"] * c["mz"], c["order"] // 2, c["visc"] // 2
    # per point: fluxes 26 and pressure 4 operations a side pair, viscous stencils, stresses, state
    flops = 3 * (30 * s + 19 * sv + 60) + 60
    if c["path"] == "rhs":
        return {"bytes": 10.0 * 8 * n, "flops": float(flops * n)}
    per = (4 if c["fp32"] else 8) * _WORDS[c["scheme"]] * n
    return {"bytes": float(per * c["steps"] + 5 * 8 * n),
            "flops": float(flops * n * _STAGES[c["scheme"]] * c["steps"])}


# ---------------------------------------------------------------------------
# the same in 64 bits with plain torch
# ---------------------------------------------------------------------------

class _Exact:
    """The flow's right-hand side and time advance on [z, y, x] tensors."""

    def __init__(self, c):
        self.c, self.cfg = c, _config(c)
        self.s, self.sv = c["order"] // 2, c["visc"] // 2
        self.g = g = _grid(c["kind"], c["mx"], c["my"], c["mz"], self.s)
        self.rg = 1.0 / (self.cfg.gam * self.cfg.Ma ** 2)
        self.cp = self.rg * self.cfg.gam / (self.cfg.gam - 1)
        self.ipe = 1.0 / (self.cfg.Pr * (self.cfg.gam - 1) * self.cfg.Ma ** 2)
        self.xp, self.xpp, self.dxv = (_t(g[k])[None, None, :] for k in ("xp", "xpp", "dxv"))
        self.h = {2: g["dx"], 1: g["dy"], 0: g["dz"]}
        self.dpdz = self.cfg.dpdz0 if self.cfg.forcing else 0.0
        self.time, self.dt, self.visc = 0.0, 0.0, None
        self.layer = c["kind"] == "layer"
        if self.layer:
            sx, sz = _layer_sponge(g)
            self.sigma = _t(sx)[None, None, :] + _t(sz)[:, None, None]
            self.ref = [_t(a)[:, None, :] for a in _layer_reference(c, g, self.cfg)]

    def mu(self, t):
        return t ** self.cfg.viscexp / self.cfg.Re

    # padding by s points along one dimension, per ghost rule
    def _wrap(self, f, d):
        n = f.shape[d]
        return torch.cat([f.narrow(d, n - self.s, self.s), f, f.narrow(d, 0, self.s)], d)

    def _low(self, f, d, sign=1.0, value=0.0):  # reflection about the lower face
        return sign * f.narrow(d, 0, self.s).flip(d) + value

    def _high(self, f, d, sign=1.0, value=0.0):
        return sign * f.narrow(d, f.shape[d] - self.s, self.s).flip(d) + value

    def _ext_high(self, f, d):  # linear extrapolation about the last node
        n = f.shape[d]
        return 2.0 * f.narrow(d, n - 1, 1) - f.narrow(d, n - 1 - self.s, self.s).flip(d)

    def _ext_low(self, f, d):
        return 2.0 * f.narrow(d, 0, 1) - f.narrow(d, 1, self.s).flip(d)

    def _blow(self, low):
        """the wall-normal blowing's u ghosts in the z planes 90..130"""
        k = np.arange(self.c["mz"])
        kap = np.where(k < 110, 1.0, -1.0)
        xi = np.where(k < 110, k - 90, 130 - k) / 20.0
        gz = kap * (15.1875 * xi ** 5 - 35.4375 * xi ** 4 + 20.25 * xi ** 3)
        on = _t(((k >= 90) & (k <= 130)).astype(float))[:, None, None]
        cosy = np.cos(np.arange(self.c["my"]) * self.g["dy"] / (self.g["L"][1] / (2 * math.pi)))
        val = (2e-4 * _t(gz)[:, None, None] * math.sin(self.cfg.Re * 121e-6 * self.time) +
               3e-5 * _t(gz)[:, None, None] * math.sin(10.0 * self.time) * _t(cosy)[None, :, None])
        return torch.where(on > 0, val.expand_as(low), low)

    def pads(self, q, d):
        """all quantities with ghosts along d (0 z, 1 y, 2 x)"""
        if d == 1 or (d == 0 and not self.layer) or (d == 2 and self.c["kind"] == "box"):
            return {k: self._wrap(f, d) for k, f in q.items()}
        if d == 0:
            return {k: torch.cat([self._ext_low(f, d), f, self._ext_high(f, d)], d) for k, f in q.items()}
        ends = {}
        for k in "uvwTpD":
            if self.layer:
                lo = self._low(q[k], d, -1.0 if k in "uvw" else 1.0)
                ends[k] = (self._blow(lo) if k == "u" else lo, self._ext_high(q[k], d))
            elif k in "uvw":
                ends[k] = (self._low(q[k], d, -1.0), self._high(q[k], d, -1.0))
            elif k == "T":
                ends[k] = (self._low(q[k], d, -1.0, 2.0 * self.cfg.twall_bot),
                           self._high(q[k], d, -1.0, 2.0 * self.cfg.twall_top))
            else:
                ends[k] = (self._low(q[k], d), self._high(q[k], d))
        for k in "rhm":
            e = []
            for i in (0, 1):
                u, v, w, t, p = (ends[x][i] for x in "uvwTp")
                e.append(p / (self.rg * t) if k == "r" else
                         (self.mu(t) if k == "m" else self.cp * t + 0.5 * (u * u + v * v + w * w)))
            ends[k] = tuple(e)
        return {k: torch.cat([ends[k][0], q[k], ends[k][1]], d) for k in q}

    def d1(self, f, d, s):
        a, n, o = _weights(s)[0], f.shape[d] - 2 * self.s, self.s
        out = sum(a[k] * (f.narrow(d, o + k, n) - f.narrow(d, o - k, n)) for k in range(1, s + 1)) / self.h[d]
        return out * self.xp if d == 2 and self.c["kind"] != "box" else out

    def d2(self, f, d):
        s, o = self.sv, self.s
        (a, b), n = _weights(s), f.shape[d] - 2 * self.s
        out = b[0] * f.narrow(d, o, n)
        for k in range(1, s + 1):
            out = out + b[k] * (f.narrow(d, o + k, n) + f.narrow(d, o - k, n))
        out = out / self.h[d] ** 2
        if d == 2 and self.c["kind"] != "box":
            first = sum(a[k] * (f.narrow(d, o + k, n) - f.narrow(d, o - k, n)) for k in range(1, s + 1)) / self.h[d]
            out = out * self.xp ** 2 - first * self.xpp * self.xp ** 3
        return out

    def flux(self, P, adv, d):
        """-D of the split forms: mass, three momenta, energy"""
        a, o, s = _weights(self.s)[0], self.s, self.s
        n = P["r"].shape[d] - 2 * s
        out = [0.0] * 5
        for l in range(1, s + 1):
            pair = lambda f: f.narrow(d, o - l, n + l) + f.narrow(d, o, n + l)  # noqa: E731
            m = pair(P["r"]) * pair(P[adv])
            for i, k in enumerate(("", "u", "v", "w", "h")):
                x = m * pair(P[k]) if k else m
                out[i] = out[i] - (0.25 if k else 0.5) * a[l] * (x.narrow(d, l, n) - x.narrow(d, 0, n))
        out = [x / self.h[d] for x in out]
        return [x * self.xp for x in out] if d == 2 and self.c["kind"] != "box" else out

    def rhs(self, q):
        r = q[0]
        u, v, w = q[1] / r, q[2] / r, q[3] / r
        k2 = 0.5 * (u * u + v * v + w * w)
        T = (q[4] / r - k2) * (self.cfg.gam - 1) / self.rg
        Q = dict(r=r, u=u, v=v, w=w, T=T, p=r * self.rg * T, h=self.cp * T + k2, m=self.mu(T))
        # velocity gradients G[component][direction] (x, y, z), then the dilatation
        dims = (2, 1, 0)
        G = [[None] * 3 for _ in range(3)]
        Q["D"] = torch.zeros_like(r)
        for j, d in enumerate(dims):
            P = self.pads(Q, d)
            for i, c in enumerate("uvw"):
                G[i][j] = self.d1(P[c], d, self.sv)
        Q["D"] = G[0][0] + G[1][1] + G[2][2]
        out = [torch.zeros_like(r) for _ in range(5)]
        mu = Q["m"]
        for j, d in enumerate(dims):
            P = self.pads(Q, d)
            S = [G[i][j] + G[j][i] if i != j else 2 * G[j][j] - 2.0 / 3.0 * Q["D"] for i in range(3)]
            # the reference's y viscous work takes dv/dz with the zy stress
            e = mu * sum(S[i] * (G[1][2] if (j == 1 and i == 2) else G[i][j]) for i in range(3))
            dm = self.d1(P["m"], d, self.sv)
            S = [S[i] * dm + mu * self.d2(P[c], d) for i, c in enumerate("uvw")]
            vel = (u, v, w)
            e = e + sum(vel[i] * S[i] for i in range(3))
            e = e + self.ipe * (mu * self.d2(P["T"], d) + self.d1(P["T"], d, self.sv) * dm)
            ac = mu * self.d1(P["D"], d, self.sv) / 3.0
            e = e + ac * vel[j]
            S[j] = S[j] + ac - self.d1(P["p"], d, self.s)
            F = self.flux(P, "uvw"[j], d)
            out[0] += F[0]
            for i in range(3):
                out[1 + i] += S[i] + F[1 + i]
            out[4] += e + F[4]
        out[3] += self.dpdz
        out[4] += self.dpdz * w
        if self.layer:
            out = [out[i] + self.sigma * (self.ref[i] - q[i]) for i in range(5)]
        return out

    def limits(self, q):
        """convective and viscous CFL maxima of a state"""
        r = q[0]
        u, v, w = q[1] / r, q[2] / r, q[3] / r
        e = q[4] / r - 0.5 * (u * u + v * v + w * w)
        gam, g = self.cfg.gam, self.g
        a = torch.sqrt(gam * (gam - 1) * e)
        conv = max(float(((u.abs() + a) / self.dxv).max()), float((v.abs() + a).max()) / g["dy"],
                   float((w.abs() + a).max()) / g["dz"])
        mu = self.mu(e * (gam - 1) / self.rg)
        visc = max(float((mu / self.dxv ** 2).max()), float(mu.max()) / g["dy"] ** 2, float(mu.max()) / g["dz"] ** 2)
        return conv, visc

    def integral(self, f):
        return float((f * self.dxv).sum()) * self.g["dy"] * self.g["dz"]

    def advance(self, f, steps):
        q = [f[0], f[0] * f[1], f[0] * f[2], f[0] * f[3], f[4]]
        cfg, add = self.cfg, lambda x, c, y: [a + c * b for a, b in zip(x, y)]
        kin, enst, time = np.full(steps, np.nan), np.full(steps, np.nan), np.zeros(steps)
        for n in range(steps):
            if n % cfg.check_cfl == 0:
                conv, here = self.limits(q)
                visc = here if self.visc is None else self.visc
                self.dt = min(1e5, cfg.cfl / max(conv, visc))
                if cfg.forcing:
                    self.dpdz = 0.99 * self.dpdz - 0.5 * (self.integral(q[3]) / self.integral(q[0]) - 1)
            self.time += self.dt
            time[n] = self.time
            if n % cfg.check_bulk == 0:
                if cfg.forcing:
                    kin[n], enst[n] = self.integral(q[3]) / self.integral(q[0]), self.integral(q[4])
                else:
                    kin[n] = self.integral(sum((m / q[0]) ** 2 for m in q[1:4])) / math.prod(self.g["L"])
            dt = self.dt
            if self.c["scheme"] == "rk3":
                prev, last = None, q
                for alpha, beta in ((0.0, 8 / 15), (-17 / 60, 5 / 12), (-5 / 12, 3 / 4)):
                    last, k = q, self.rhs(q)
                    q = add(q, dt * beta, k)
                    q = add(q, dt * alpha, prev) if prev is not None else q
                    prev = k
            elif self.c["scheme"] == "kutta_rk3":
                k1 = self.rhs(q)
                k2 = self.rhs(add(q, dt / 2, k1))
                last = add(add(q, 2 * dt, k2), -dt, k1)
                k3 = self.rhs(last)
                q = add(add(add(q, dt / 6, k1), 4 * dt / 6, k2), dt / 6, k3)
            else:
                k = self.rhs(q)
                acc, last = add(q, dt / 6, k), add(q, dt / 2, k)
                k = self.rhs(last)
                acc, last = add(acc, dt / 3, k), add(q, dt / 2, k)
                k = self.rhs(last)
                acc, last = add(acc, dt / 3, k), add(q, dt, k)
                q = add(acc, dt / 6, self.rhs(last))
            if (n + 1) % cfg.check_cfl == 0:
                self.visc = self.limits(last)[1]  # the viscous limit lags by one stage
        return q, kin, enst, time

    def profiles(self, q):
        """wall-normal profiles: plane means, Favre velocities, mean squared deviations"""
        plane = lambda f: f.mean(dim=(0, 1))  # noqa: E731
        r = plane(q[0])
        um = [plane(q[i]) / r for i in (1, 2, 3)]
        em = plane(q[4])
        dev = [plane((q[0] - r) ** 2)] + [plane((q[i] / q[0] - um[i - 1]) ** 2) for i in (1, 2, 3)]
        cols = [_t(self.g["x"]), r, *um, em, *dev, plane((q[4] - em) ** 2)]
        return {k: a.cpu() for k, a in zip(cns.Solver.PROFILE_COLUMNS, cols)}


def _exact_cost(c):
    n = 1 if c["path"] == "rhs" else c["steps"] * _STAGES[c["scheme"]]
    return n * c["mx"] * c["my"] * c["mz"] * (2.0 + 0.5 * c["order"])


def exact(case, seed):
    c = dict(case)
    if c["path"] == "batch":
        cs = _members(c, seed)
        if sum(map(_exact_cost, cs)) > 1.8e10:
            return None
        out = []
        for k, m in enumerate(cs):
            q = _Exact(m).advance(_fields(m, seed * 131 + k), m["steps"])[0]
            out.append([q[0].reshape(-1)] + [(a / q[0]).reshape(-1) for a in q[1:4]] + [q[4].reshape(-1)])
        return out
    if _exact_cost(c) > 1.8e10:
        return None
    X, f = _Exact(c), _fields(c, seed)
    if c["path"] == "rhs":
        return torch.stack(X.rhs([f[0], f[0] * f[1], f[0] * f[2], f[0] * f[3], f[4]]))
    q, kin, enst, time = X.advance(f, c["steps"])
    out = dict(kin=kin, enst=enst, time=time,
               state=[q[0].reshape(-1)] + [(a / q[0]).reshape(-1) for a in q[1:4]] + [q[4].reshape(-1)])
    if c["kind"] == "channel":
        out.update(X.profiles(q))
    return out
