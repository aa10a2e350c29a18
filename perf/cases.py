"""The soap-film step's measured cases: what a program that uses this library has
it do, over the sizes, precisions and options it is used with.

Every case is a running simulation: a handle (or, for the entry point without
allocation, device arrays) that holds one or more films, and a pass that
advances it by a number of steps and takes the result back: the whole state,
or, for a frame, the thickness image. The sizes, steps and parameters are those
of the repository's configurations, tests and benchmark: 64x128, 256x512 and
1024x2048 films, the uneven batch of 96 bubbles, the 2048x4096 bubbles of the
large batch, grids that are no power of two, and the reference's own
config.txt regime.

A case's fields:
  kind     "film" (one bubble or several of one handle, the state comes back),
           "frame" (the frame loop: steps, then the thickness image),
           "device" (steps on device-resident arrays)
  sizes    n_theta of each group of bubbles, comma-separated; `counts` how many
           of each; n_phi = 2 n_theta; `dts` the step of each group, in seconds
  steps    steps of one pass
  prec     "mixed" (FP32 fields, FP64 refinement) or "fp64"
  radius   m; with gravity and evaporation where `driver` is true, as the
           command-line driver sets them (its solves stop at an absolute 1e-7)
  scalar   "plain" or "bimocq" advection of the thickness
"""
import math

import numpy as np
import torch

import soapbubble_amd as sb

FIELDS = ("u_theta", "u_phi", "eta", "gamma")
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
T_AIR = 0.5      # air-flow time of every pass, in seconds (held, as the frame loop holds it)
F64 = torch.float64


def _case(name, kind, sizes, counts, dts, steps, prec="mixed", radius=1.0, driver=False,
          scalar="plain", noise=0.0, l_max=16):
    c = {"kind": kind, "sizes": sizes, "counts": counts, "dts": dts, "steps": steps, "prec": prec,
         "radius": radius, "driver": driver, "scalar": scalar, "noise": noise, "l_max": l_max}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest film, in double precision: a quick look at a coarse grid,
        # all latency and launches
        _case("film 64x128 fp64", "film", "64", "1", "0.005", 20, prec="fp64", l_max=4),
        # an ordinary film, replayed as graphs: 131 072 cells
        _case("film 256x512", "film", "256", "1", "0.002", 100),
        # the reference's resolution class and the benchmark's headline film
        _case("film 1024x2048", "film", "1024", "1", "0.001", 100, noise=0.05, l_max=64),
        # the same film on the plain double-precision path
        _case("film 1024x2048 fp64", "film", "1024", "1", "0.001", 20, prec="fp64", noise=0.05,
              l_max=64),
        # a grid that is no power of two, as numberOfGridsInTheta may be anything
        _case("film 1000x2000", "film", "1000", "1", "0.001", 50, l_max=64),
        # a small odd grid
        _case("film 101x202", "film", "101", "1", "0.004", 50),
        # the largest film
        _case("film 2048x4096", "film", "2048", "1", "0.0005", 40, l_max=128),
        # the uneven batch of 96 bubbles advanced together
        _case("batch 96 bubbles", "film", "64,128,256", "32,32,32", "0.005,0.004,0.002", 200),
        # one frame of the frame loop with its thickness image
        _case("frame 1024x2048", "frame", "1024", "1", "0.001", 10, l_max=32),
        # the driver's default scalar advection (BIMOCQ with its five samples)
        _case("bimocq 512x1024", "film", "512", "1", "0.0001", 20, radius=0.05, driver=True,
              scalar="bimocq"),
        # the reference's config.txt (radius 0.05 m, 0.005 s a step, four steps a
        # frame): the stiff regime, where the solve takes multigrid
        _case("config.txt 256x512", "film", "256", "1", "0.005", 4, radius=0.05, driver=True),
        # steps on device-resident arrays without any allocation
        _case("device 128x256", "device", "128", "1", "0.004", 20),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("film", "film", "film", "fp64", "batch", "frame", "bimocq", "stiff", "device"))
    steps = rng.randint(10, 60)

    def dt(n):
        return "%.3g" % min(0.005, rng.uniform(0.5, 1.0) / n)

    if kind == "batch":
        sizes = sorted(_logint(rng, 24, 220) for _ in range(3))
        return _case("", "film", ",".join(map(str, sizes)),
                     ",".join(str(rng.randint(1, 10)) for _ in sizes),
                     ",".join(dt(n) for n in sizes), steps)
    if kind == "stiff":   # the config.txt regime around its own resolution
        n = 16 * rng.randint(6, 20)
        return _case("", "film", str(n), "1", "0.005", rng.randint(2, 6), radius=0.05, driver=True)
    if kind == "bimocq":
        n = _logint(rng, 48, 640)
        return _case("", "film", str(n), "1", "%.3g" % (0.05 * rng.uniform(0.5, 1.2) / n),
                     rng.randint(8, 20), radius=0.05, driver=True, scalar="bimocq")
    if kind == "device":
        n = _logint(rng, 24, 360)
        return _case("", "device", str(n), "1", dt(n), rng.randint(5, 30))
    if kind == "fp64":
        n = _logint(rng, 24, 900)
        return _case("", "film", str(n), "1", dt(n), rng.randint(4, 16), prec="fp64")
    if kind == "frame":
        n = _logint(rng, 64, 1024)
        return _case("", "frame", str(n), "1", dt(n), rng.randint(4, 16))
    n = _logint(rng, 32, 1024)
    return _case("", "film", str(n), "1", dt(n), steps, noise=rng.choice((0.0, 0.05)))


# ------------------------------------------------------------------ inputs ----
def _bubbles(case):
    """(n_theta, dt) of every bubble of the case, in order."""
    out = []
    for n, k, dt in zip(case["sizes"].split(","), case["counts"].split(","), case["dts"].split(",")):
        out += [(int(n), float(dt))] * int(k)
    return out


def _waves(gen, l_max, th, ph):
    """A smooth field on the sphere: 16 plane waves of wave number up to l_max
    restricted to the points (th, ph), scaled to a largest value of 1."""
    r = np.asarray(gen.normal(size=(16, 3)))
    k = r / np.linalg.norm(r, axis=1, keepdims=True) * gen.uniform(1.0, l_max, size=(16, 1))
    a, p = gen.uniform(-1, 1, 16), gen.uniform(0, 2 * np.pi, 16)
    st, ct = torch.sin(th)[:, None], torch.cos(th)[:, None]
    x, y, z = st * torch.cos(ph)[None], st * torch.sin(ph)[None], ct.expand(len(th), len(ph))
    f = torch.zeros_like(x)
    for q in range(16):
        f += float(a[q]) * torch.cos(float(k[q, 0]) * x + float(k[q, 1]) * y + float(k[q, 2]) * z +
                                     float(p[q]))
    return f


def _inputs(case, seed, b, n):
    """Bubble b's initial state, air flow and Marangoni scale (FP64): a film with
    smooth thickness and concentration (and, with noise, cell-scale thickness
    variations), at rest, in a divergence-free air flow."""
    gen = np.random.default_rng([int(seed), b])
    m, h = 2 * n, math.pi / n
    ar = lambda k, o: (torch.arange(k, dtype=F64, device=DEVICE) + o) * h
    unit = lambda f: f / f.abs().max()
    many = "," in case["counts"] or case["counts"] != "1"
    amp, ms = (gen.uniform(0.2, 1.0), gen.uniform(0.5, 2.0)) if many else (1.0, 1.0)
    eta = 1.0 + 0.1 * unit(_waves(gen, case["l_max"], ar(n, 0.5), ar(m, 0.0)))
    if case["driver"]:
        eta = 0.5 * eta          # the driver's film around its default thickness
        amp *= case["radius"]    # and air flow scaled by the radius
    if case["noise"]:
        eta += case["noise"] * torch.from_numpy(gen.uniform(-1, 1, (n, m))).to(DEVICE)
    gam = 1.0 + 0.05 * unit(_waves(gen, case["l_max"], ar(n, 0.5), ar(m, 0.0)))
    psi = _waves(gen, 8.0, ar(n + 1, 0.0), ar(m, -0.5))
    psi[0], psi[n] = psi[0, 0].clone(), psi[n, 0].clone()
    ua = (psi[1:] - psi[:-1]) / h
    va = -(torch.roll(psi[1:n], -1, 1) - psi[1:n]) / (h * torch.sin(ar(n - 1, 1.0)))[:, None]
    s = amp / max(float(ua.abs().max()), float(va.abs().max()))
    return {"u_theta": torch.zeros(n - 1, m, dtype=F64, device=DEVICE),
            "u_phi": torch.zeros(n, m, dtype=F64, device=DEVICE), "eta": eta, "gamma": gam,
            "uair0": ua * s, "vair0": va * s, "M_scale": float(ms)}


def _desc(case, n, dt, ms):
    d = case["driver"]
    return sb.bubble(n, dt, radius=case["radius"], gravity=d, evaporation=d, M_scale=ms)


def prepare(case, seed):
    bub = _bubbles(case)
    ins = [_inputs(case, seed, b, n) for b, (n, _) in enumerate(bub)]
    if case["kind"] == "device":
        n, dt = bub[0]
        dev = {k: ins[0][k].float().contiguous() for k in FIELDS + ("uair0", "vair0")}
        return {"case": case, "in": dev, "out": {k: torch.empty_like(dev[k]) for k in FIELDS},
                "bubble": _desc(case, n, dt, ins[0]["M_scale"]),
                "opt": sb.options("mixed", advance_time=False)}
    ctx = sb.SoapFilm([_desc(case, n, dt, i["M_scale"]) for (n, dt), i in zip(bub, ins)],
                      case["prec"], use_graph=case["prec"] == "mixed", advance_time=False,
                      tol=1e-7 if case["driver"] else 1e-10, tol_absolute=bool(case["driver"]),
                      scalar_advection=case["scalar"])
    for b, i in enumerate(ins):
        for k in FIELDS + ("uair0", "vair0"):
            ctx.upload(b, k, i[k].cpu().numpy())
    ctx.set_time(T_AIR)
    return {"case": case, "ctx": ctx, "bubbles": len(bub)}


def run(state):
    case = state["case"]
    if case["kind"] == "device":
        i, o = state["in"], state["out"]
        sb.step_noalloc(state["bubble"], state["opt"], T_AIR, case["steps"],
                        [i[k].data_ptr() for k in FIELDS],
                        [i["uair0"].data_ptr(), i["vair0"].data_ptr()],
                        [o[k].data_ptr() for k in FIELDS],
                        torch.cuda.current_stream().cuda_stream)
        return o
    ctx = state["ctx"]
    if case["kind"] == "frame":
        ctx.set_time(T_AIR)
        ctx.step(case["steps"])
        return ctx.thickness_half(0).view(np.float16)
    ctx.step(case["steps"])
    # the mixed paths' fields are FP32, handed over as doubles
    ty = np.float64 if case["prec"] == "fp64" else np.float32
    if state["bubbles"] == 1:
        return {k: ctx.download(0, k).astype(ty, copy=False) for k in FIELDS}
    return {k: np.concatenate([ctx.download(b, k) for b in range(state["bubbles"])], dtype=ty,
                              casting="same_kind") for k in FIELDS}


def work(case):
    """Per step: the state read and written once and the air flow read once, the
    arithmetic of three back-traces, one five-point system and the updates; once
    a pass, the result."""
    cells = sum(2 * n * n for n, _ in _bubbles(case))
    size = 8 if case["prec"] == "fp64" else 4
    per = {"plain": 1500, "bimocq": 9000}[case["scalar"]]
    out = 2 if case["kind"] == "frame" else 4 * size
    return {"bytes": cells * (case["steps"] * 10 * size + out), "flops": cells * case["steps"] * per}


# ------------------------------------------------------- the step in FP64 ----
# The same step in plain torch, in double precision throughout, for a group of
# bubbles of one size: fields are (bubbles, rows, columns).
class _Grid:
    def __init__(self, n, dts, ms, case):
        self.n, self.m, self.h = n, 2 * n, math.pi / n
        R, T, H, gm = 8.3144598, 298.15, 1e-6, 1e-6
        rad = case["radius"]
        col = lambda v: torch.tensor(v, dtype=F64, device=DEVICE).reshape(-1, 1, 1)
        self.dt = col([d / rad for d in dts])
        self.M = col([gm * R * T / (3e3 * H) * s for s in ms])
        self.Cr = 1.184 * math.sqrt(1.562e-5 * rad) / (1e3 * H)
        self.gs = 9.8 * rad if case["driver"] else 0.0
        self.eva = -3e-8 * rad / H if case["driver"] else 0.0
        self.gmax = 0.07275 / (R * T) / gm
        ar = lambda k, o: torch.arange(k, dtype=F64, device=DEVICE) + o
        self.tc, self.tf = ar(n, 0.5)[:, None], ar(n - 1, 1.0)[:, None]
        self.pc, self.ph = ar(self.m, 0.0)[None], ar(self.m, -0.5)[None]
        self.sc = torch.sin(self.tc * self.h)
        self.sf = torch.sin(ar(n + 1, 0.0)[:, None] * self.h)
        self.sf[0] = self.sf[n] = 0.0
        self.kt = 3.0 - abs(T_AIR - 3.0)
        # the air corridor: a band around the great circle normal to -y, its
        # speed 0.5 sin(beta) radius faded by smoothstep(0.2, 0.4, |beta - pi/2|)
        def corridor(t, p, phi_part):
            t, p = t * self.h, p * self.h
            w = (torch.sin(t) * torch.cos(p), torch.sin(t) * torch.sin(p), torch.cos(t) + 0 * p)
            nrm = torch.tensor([0.0, -math.sin(math.pi / 2), math.cos(math.pi / 2)], dtype=F64)
            nx, ny, nz = (float(v) for v in nrm / nrm.norm())
            c = (nx * w[0] + ny * w[1] + nz * w[2]).clamp(-1, 1)
            q = [w[k] - c * v for k, v in enumerate((nx, ny, nz))]
            inv = 1.0 / torch.sqrt(q[0] ** 2 + q[1] ** 2 + q[2] ** 2)
            q = [v * inv for v in q]
            x = (ny * q[2] - nz * q[1], nz * q[0] - nx * q[2], nx * q[1] - ny * q[0])
            beta = torch.acos(c)
            y = ((beta - math.pi / 2).abs().float() - 0.2) / (torch.tensor(0.4) - 0.2).item()
            y = y.clamp(0, 1)
            s = (1.0 - (y * y * (3.0 - 2.0 * y)).double()) * 0.5 * torch.sin(beta) * rad
            if phi_part:
                return s * (-torch.sin(p) * x[0] + torch.cos(p) * x[1])
            return s * (torch.cos(t) * (torch.cos(p) * x[0] + torch.sin(p) * x[1]) -
                        torch.sin(t) * x[2])
        self.au = corridor(self.tc, self.ph, True)
        self.av = corridor(self.tf, self.pc, False)

    def centred(self, f):    # with a row beyond each pole: the cells at phi + pi
        s = lambda r: torch.roll(r, self.n, -1)
        return torch.cat((s(f[:, :1]), f, s(f[:, -1:])), 1)

    def vphi(self, f):
        s = lambda r: -torch.roll(r, self.n, -1)
        return torch.cat((s(f[:, :1]), f, s(f[:, -1:])), 1)

    def vtheta(self, f):     # with the pole rows: the mean across the pole
        s = lambda r: 0.5 * (r - torch.roll(r, self.n, -1))
        return torch.cat((s(f[:, :1]), f, s(f[:, -1:])), 1)

    def corners(self, x, y, rows):
        fx, fy = torch.floor(x).clamp(0, rows - 2), torch.floor(y)
        i = fx.long() * self.m
        c0 = torch.remainder(fy.long(), self.m)
        c1 = torch.remainder(c0 + 1, self.m)
        return (i + c0, i + c1, i + self.m + c0, i + self.m + c1), x - fx, y - fy

    def at(self, f, k):
        return torch.gather(f.flatten(1), 1, k.flatten(1)).view(k.shape)

    def bilinear(self, f, x, y):
        k, a, b = self.corners(x, y, f.shape[1])
        lo = (1 - b) * self.at(f, k[0]) + b * self.at(f, k[1])
        hi = (1 - b) * self.at(f, k[2]) + b * self.at(f, k[3])
        return (1 - a) * lo + a * hi

    def s_centred(self, f, t, p):
        return self.bilinear(f, t + 0.5, p)

    def s_vphi(self, f, t, p):
        return self.bilinear(f, t + 0.5, p + 0.5)

    def s_vtheta(self, f, t, p):
        return self.bilinear(f, t, p)


def _cross(a, b):
    return (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _index(g, p):
    return torch.atan2(torch.sqrt(p[0] ** 2 + p[1] ** 2), p[2]) / g.h, torch.atan2(p[1], p[0]) / g.h


def _frame(t, p, g):
    """e_theta, e_phi and the unit vector of the point with index coordinates (t, p)."""
    st, ct = torch.sin(t * g.h), torch.cos(t * g.h)
    sp, cp = torch.sin(p * g.h), torch.cos(p * g.h)
    zero = 0 * (st * sp)
    return (ct * cp, ct * sp, -st + zero), (-sp + zero, cp + zero, zero), (st * cp, st * sp, ct + zero)


def _carry(g, uth, uph, w, d, speed, dt):
    """The velocity at the point `dt` of motion along -d from w, carried along the
    great circle back to w: (its component along d, across d), and the point."""
    s, c = torch.sin(-speed * dt), torch.cos(-speed * dt)
    q = tuple(d[k] * s + w[k] * c for k in range(3))
    t, p = _index(g, q)
    vt, vp = g.s_vtheta(uth, t, p), g.s_vphi(uph, t, p)
    et, ep, _ = _frame(t, p, g)
    v = tuple(vt * et[k] + vp * ep[k] for k in range(3))
    along = tuple(d[k] * c - w[k] * s for k in range(3))
    return _dot(v, along), _dot(v, _cross(q, along)), t, p


def _trace(g, uth, uph, t, p, ut, up, dt):
    """The great-circle back-trace from the points (t, p) with velocity (ut, up):
    the departure point and the velocity there carried back to the start."""
    et, ep, w = _frame(t, p, g)
    u = tuple(ut * et[k] + up * ep[k] for k in range(3))
    speed = torch.sqrt(_dot(u, u))
    safe = torch.where(speed > 0, speed, torch.ones_like(speed))
    d = tuple(v / safe for v in u)
    a, b, _, _ = _carry(g, uth, uph, w, d, speed, 0.5 * dt)
    v = _cross(w, d)
    mid = tuple(a * d[k] + b * v[k] for k in range(3))
    s2 = torch.sqrt(_dot(mid, mid))
    moving = (speed > 0) & (s2 > 0)
    safe = torch.where(moving, s2, torch.ones_like(s2))
    d = tuple(m / safe for m in mid)
    a, b, dt_, dp_ = _carry(g, uth, uph, w, d, s2, dt)
    v = _cross(w, d)
    back = tuple(torch.where(moving, a * d[k] + b * v[k], torch.zeros_like(a)) for k in range(3))
    one = torch.ones_like(a)
    return (torch.where(moving, dt_, t * one), torch.where(moving, dp_, p * one), _dot(back, et),
            _dot(back, ep))


def _centre_velocity(g, uth, uph):
    return (g.s_vtheta(uth, *_grid(g, uth, g.tc, g.pc)), g.s_vphi(uph, *_grid(g, uph, g.tc, g.pc)))


def _grid(g, f, t, p):
    one = torch.ones(f.shape[0], t.shape[0], p.shape[1], dtype=F64, device=DEVICE)
    return t * one, p * one


class _Line:
    """The periodic tridiagonal phi systems -w x_{i-1} + d x_i - e x_{i+1} of every
    row, factored by cyclic reduction (whose couplings fall below rounding)."""

    def __init__(self, w, d, e):
        a, c = -w / d, -e / d
        self.inv, self.level, s = 1.0 / d, [], 1
        while float(torch.maximum(a.abs().max(), c.abs().max())) > 1e-18 and len(self.level) < 40:
            am, cm = torch.roll(a, s, -1), torch.roll(c, s, -1)
            ap, cp = torch.roll(a, -s, -1), torch.roll(c, -s, -1)
            k = 1.0 / (1.0 - a * cm - c * ap)
            self.level.append((s, a * k, c * k, k))
            a, c = -a * am * k, -c * cp * k
            s = (2 * s) % w.shape[-1]
            if s == 0:    # every cell is coupled to itself alone
                break
        self.last = 1.0 / (1.0 + a + c) if s == 0 else None

    def __call__(self, r):
        x = r * self.inv
        for s, a, c, k in self.level:
            x = k * x - a * torch.roll(x, s, -1) - c * torch.roll(x, -s, -1)
        return x if self.last is None else x * self.last


def _solve(wn, ws, ww, we, dg, b, x):
    """Conjugate gradients with the phi-line preconditioner to 1e-13."""
    line = _Line(ww, dg, we)
    z_row = torch.zeros_like(x[:, :1])

    def A(v):
        y = dg * v - ww * torch.roll(v, 1, -1) - we * torch.roll(v, -1, -1)
        return y - wn * torch.cat((z_row, v[:, :-1]), 1) - ws * torch.cat((v[:, 1:], z_row), 1)

    sm = lambda u, v: (u * v).sum((1, 2), keepdim=True)
    r = b - A(x)
    bb = sm(b, b)
    z = line(r)
    p, rz = z, sm(r, z)
    for it in range(1500):
        q = A(p)
        a = rz / sm(p, q)
        x, r = x + a * p, r - a * q
        if it % 4 == 3 and bool((sm(r, r) <= 1e-26 * bb).all()):
            break
        z = line(r)
        new = sm(r, z)
        p, rz = z + (new / rz) * p, new
    return x


def _body(g, S, air):
    """Assembly, solve and updates from the advected state S; the new state."""
    ut, up, eta, gam = (S[k] for k in FIELDS)
    h, dt, Cr, M = g.h, g.dt, g.Cr, g.M
    ua, va = air["uair0"] + g.au * g.kt, air["vair0"] + g.av * g.kt
    mir = lambda f: torch.roll(f.flip(-1), 1, -1)
    bl = T_AIR / 12.0
    uab, vab = 0.5 * (ua * bl + mir(ua) * (1 - bl)), 0.5 * (va * bl - mir(va) * (1 - bl))
    zr = torch.zeros_like(eta[:, :1])
    west = lambda f: torch.roll(f, 1, -1)
    east = lambda f: torch.roll(f, -1, -1)
    fw = 0.5 * (west(eta) + eta)                                   # west faces
    fn = torch.cat((zr, 0.5 * (eta[:, :-1] + eta[:, 1:]), zr), 1)  # faces 0..n
    kw, kn = 1.0 / (fw + Cr * dt), 1.0 / (fn + Cr * dt)
    s2 = 1.0 / (h * h)
    ww = s2 / g.sc * M * dt * kw
    wf = s2 * g.sf * M * dt * kn
    wn, ws = wf[:, :-1], wf[:, 1:]
    flux = g.sf * torch.cat((zr, ut, zr), 1) * fn * kn
    flux = flux + Cr * dt * g.sf * torch.cat((zr, vab, zr), 1) * kn
    flux = flux + g.gs * dt * g.sf * g.sf * fn * kn
    fphi = up * fw * kw + Cr * dt * uab * kw
    div = (east(fphi) - fphi + flux[:, 1:] - flux[:, :-1]) / h
    dg = g.sc / dt / gam + wn + ws + ww + east(ww)
    x = _solve(wn, ws, ww, east(ww), dg, g.sc / dt - div, gam)
    new = torch.where((x <= 0) | (x > g.gmax - 1e-7), torch.full_like(x, g.gmax), x)
    div = (1.0 - torch.minimum(x, 2 * gam) / gam) / dt
    e1 = torch.clamp(eta * (1 - dt * div) + g.eva * dt, min=0.0)
    ie = 1.0 / fw
    u1 = (up / dt - M * ie * (new - west(new)) / h / g.sc + Cr * ie * ua) / (1.0 / dt + Cr * ie)
    ie = 1.0 / fn[:, 1:-1]
    v1 = (ut / dt - M * ie * (new[:, 1:] - new[:, :-1]) / h + Cr * ie * va + g.gs * g.sf[1:-1]) / (
        1.0 / dt + Cr * ie)
    return {"u_theta": v1, "u_phi": u1, "eta": e1, "gamma": new}


def _advect(g, S):
    uth, uph = g.vtheta(S["u_theta"]), g.vphi(S["u_phi"])
    ct, cp = _centre_velocity(g, uth, uph)
    t, p, _, _ = _trace(g, uth, uph, g.tc, g.pc, ct, cp, g.dt)
    out = {k: g.s_centred(g.centred(S[k]), t, p) for k in ("eta", "gamma")}
    gt = g.s_vtheta(uth, *_grid(g, uth, g.tc, g.ph))
    out["u_phi"] = _trace(g, uth, uph, g.tc, g.ph, gt, S["u_phi"], g.dt)[3]
    gp = g.s_vphi(uph, *_grid(g, uph, g.tf, g.pc))
    out["u_theta"] = _trace(g, uth, uph, g.tf, g.pc, S["u_theta"], gp, g.dt)[2]
    return out


def _slerp(f, t, a):
    c = _dot(f, t).clamp(-1, 1)
    k = _cross(f, t)
    th = torch.atan2(torch.sqrt(_dot(k, k)), c)
    s = torch.sin(th)
    same = s == 0
    s = torch.where(same, torch.ones_like(s), s)
    u = torch.where(same, torch.ones_like(s), torch.sin((1 - a) * th) / s)
    v = torch.where(same, torch.zeros_like(s), torch.sin(a * th) / s)
    return tuple(u * f[q] + v * t[q] for q in range(3))


def _lookup(g, M, t, p):
    """The map M (unit vectors) at the points (t, p), by spherical interpolation."""
    E = [g.centred(c) for c in M]
    k, a, b = g.corners(t + 0.5, p, E[0].shape[1])
    v = [tuple(g.at(e, q) for e in E) for q in k]
    return _slerp(_slerp(v[0], v[1], b), _slerp(v[2], v[3], b), a)


_MS = ((0.125, -0.25, -0.25), (0.125, 0.25, -0.25), (0.125, -0.25, 0.25), (0.125, 0.25, 0.25),
       (0.5, 0.0, 0.0))


def _bimocq(g, S, air, steps):
    """Steps with the BIMOCQ thickness advection from a fresh start; None once the
    maps drift as far as a reinitialisation."""
    one = torch.ones_like(S["eta"])
    t0, p0 = g.tc * one, g.pc * one
    start = _frame(t0, p0, g)[2]
    fwd, bwd, prev = start, start, start
    init = last = S["eta"]
    delta = torch.zeros_like(one)
    for _ in range(steps):
        uth, uph = g.vtheta(S["u_theta"]), g.vphi(S["u_phi"])
        ct, cp = _centre_velocity(g, uth, uph)
        new = [_lookup(g, m, *_trace(g, uth, uph, g.tc, g.pc, ct, cp, s * g.dt)[:2])
               for m, s in ((fwd, -1.0), (bwd, 1.0))]
        fwd, bwd = new
        star = _advect(g, S)
        acc = torch.zeros_like(one)
        cd, ci, cl = (g.centred(f) for f in (delta, init, last))
        for w, dx, dy in _MS:
            ip = _index(g, _lookup(g, bwd, t0 + dx, p0 + dy))
            lp = _index(g, _lookup(g, prev, *ip))
            d = g.s_centred(cd, *ip)
            acc += 0.5 * w * (g.s_centred(cl, *lp) + d)
            acc += 0.5 * w * (g.s_centred(ci, *ip) + d)
        star["eta"] = acc.clamp(min=0.0)
        S = _body(g, star, air)
        chg = g.centred(S["eta"] - star["eta"])
        for w, dx, dy in _MS:
            delta = delta + w * g.s_centred(chg, *_index(g, _lookup(g, fwd, t0 + dx, p0 + dy)))
        far = 0.0
        for a, b in ((fwd, bwd), (bwd, fwd)):
            q = _lookup(g, b, *_index(g, a))
            far = max(far, float((torch.acos(_dot(q, start).clamp(-1, 1)) / g.h).max()))
        if far > 3.5:
            return None
    return S


def exact(case, seed):
    bub = _bubbles(case)
    got, b = {k: [] for k in FIELDS}, 0
    while b < len(bub):
        n = bub[b][0]
        group = [q for q in range(len(bub)) if bub[q][0] == n and q >= b]
        b = group[-1] + 1
        ins = [_inputs(case, seed, q, n) for q in group]
        g = _Grid(n, [bub[q][1] for q in group], [i["M_scale"] for i in ins], case)
        S = {k: torch.stack([i[k] for i in ins]) for k in FIELDS}
        air = {k: torch.stack([i[k] for i in ins]) for k in ("uair0", "vair0")}
        if case["scalar"] == "bimocq":
            S = _bimocq(g, S, air, case["steps"])
            if S is None:
                return None
        else:
            for _ in range(case["steps"]):
                S = _body(g, _advect(g, S), air)
        if case["kind"] == "frame":
            return (S["eta"][0] * 1e-6 * 2e5).cpu().numpy()
        for k in FIELDS:
            got[k].append(S[k].flatten().cpu().numpy())
    out = {k: np.concatenate(v) for k, v in got.items()}
    if case["kind"] == "device":
        n = bub[0][0]
        return {k: v.reshape(-1, 2 * n) for k, v in out.items()}
    return out
