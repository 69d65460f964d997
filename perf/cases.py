"""Performance cases of the spherical-fluid time step, through the entry points
a user's program calls:

  entry "noalloc"  kam_sim_step_noalloc: full steps of one sphere whose fields
                   are the caller's own device buffers
  entry "frame"    Sim.step(n) and the read-back of the frame: what the
                   configKamino.txt driver does for every frame it writes
  entry "engine"   an Engine full of resident simulations, in which requests
                   join, run their steps in the shared steps and leave with
                   their fields: batching and serving

Sizes are those of the benchmark, the driver's default and the tests, and other
supported ones (2^a 3^b 5^c) between them; dt = 0.5 / n_theta throughout.
Inputs are seeded flows of the benchmark's kind: the discrete curl of a random
spherical-harmonic streamfunction, a density band with seeded noise.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

import kaminogpu_amd as K

# every supported n_theta the drawn cases pick from
SIZES = [n for n in range(16, 2049) if n // math.gcd(n, 2 ** 11 * 3 ** 6 * 5 ** 4) == 1]


def listed():
    return [
        # the smallest call: one step of a small sphere in a caller's tight loop (latency and launches count)
        {"name": "noalloc_32", "entry": "noalloc", "nt": 32, "steps": 1, "fp64": False, "geometric": True,
         "density": True},
        # a small ragged sphere (3 5^2: an odd half spectrum) without the metric term, velocities only
        {"name": "noalloc_75_plain", "entry": "noalloc", "nt": 75, "steps": 3, "fp64": False, "geometric": False,
         "density": False},
        # the benchmark's sphere size on device-resident fields
        {"name": "noalloc_256", "entry": "noalloc", "nt": 256, "steps": 8, "fp64": False, "geometric": True,
         "density": True},
        # an odd size near the largest this entry holds, with the FP64 pressure
        {"name": "noalloc_405_fp64", "entry": "noalloc", "nt": 405, "steps": 4, "fp64": True, "geometric": True,
         "density": True},
        # the driver's default configuration: one frame of a 128 x 256 sphere with particles (density 25)
        {"name": "frame_128_particles", "entry": "frame", "nt": 128, "steps": 9, "particles": 819200, "fp64": False},
        # one frame of the benchmark's plain sphere (dt 0.002, 24 frames a second)
        {"name": "frame_256", "entry": "frame", "nt": 256, "steps": 21, "particles": 0, "fp64": False},
        # one frame of the benchmark's large sphere
        {"name": "frame_1024", "entry": "frame", "nt": 1024, "steps": 43, "particles": 0, "fp64": False},
        # the largest supported sphere
        {"name": "frame_2048", "entry": "frame", "nt": 2048, "steps": 64, "particles": 0, "fp64": False},
        # the benchmark's batch: 128 spheres of 256 x 512 in three groups with 32-step graphs, 8 of them new
        {"name": "batch_256", "entry": "engine", "lo": 256, "hi": 256, "residents": 120, "requests": 8, "steps": 96,
         "fp64": False, "graph": True},
        # the same spheres with the FP64 pressure, fewer of them
        {"name": "batch_256_fp64", "entry": "engine", "lo": 256, "hi": 256, "residents": 44, "requests": 4,
         "steps": 64, "fp64": True, "graph": True},
        # the benchmark's uneven batch of 64 spheres, requests of different lengths, direct launches
        {"name": "uneven_32_256", "entry": "engine", "lo": 32, "hi": 256, "residents": 56, "requests": 8,
         "steps": 48, "fp64": False, "graph": False},
        # the serving mix: sizes over [32, 512], requests of different lengths, direct launches
        {"name": "served_32_512", "entry": "engine", "lo": 32, "hi": 512, "residents": 84, "requests": 12,
         "steps": 40, "fp64": False, "graph": False},
    ]


def _size(rng, lo, hi):
    """A supported size, log-uniform in [lo, hi]."""
    x = math.log(lo) + rng.random() * (math.log(hi) - math.log(lo))
    return min((n for n in SIZES if lo <= n <= hi), key=lambda n: abs(math.log(n) - x))


def draw(rng):
    entry = rng.choice(["noalloc", "noalloc", "frame", "frame", "engine"])
    if entry == "noalloc":
        return {"entry": entry, "nt": _size(rng, 24, 512), "steps": rng.randint(1, 12), "fp64": rng.random() < 0.25,
                "geometric": rng.random() < 0.8, "density": rng.random() < 0.8}
    if entry == "frame":
        fp64 = rng.random() < 0.25
        nt = _size(rng, 48, 1024 if fp64 else 2048)
        steps = max(4, min(64, int(nt / 24 * (0.6 + 0.8 * rng.random()))))
        particles = rng.randint(1000, 1000000) if rng.random() < 0.3 else 0
        return {"entry": entry, "nt": nt, "steps": steps, "particles": particles, "fp64": fp64}
    lo = _size(rng, 32, 256)
    hi = lo if rng.random() < 0.4 else _size(rng, lo, 512)
    # at most half the cells of the listed batch
    count = max(4, min(160, int(64 * 256 ** 2 / (lo * hi))))
    residents = rng.randint(max(3, count // 2), count)
    return {"entry": entry, "lo": lo, "hi": hi, "residents": residents, "requests": rng.randint(1, 8),
            "steps": rng.randint(16, 64), "fp64": rng.random() < 0.25, "graph": rng.random() < 0.4}


def _members(case):
    """(n_theta, steps) of an engine case's requests and the sizes of its residents; fixed by the case."""
    rng = random.Random(1000 * case["lo"] + case["hi"])
    requests = []
    for _ in range(case["requests"]):
        nt = _size(rng, case["lo"], case["hi"])
        # with graphs a job of equal lengths; in a serving mix each request has its own
        requests.append((nt, case["steps"] if case["graph"] else rng.randint(case["steps"] // 2, case["steps"])))
    return requests, [_size(rng, case["lo"], case["hi"]) for _ in range(case["residents"])]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _fields(nt, seed):
    """Seeded FP32 (u_phi, u_theta, rho): the discrete curl, at cell corners, of
    psi = sum c_lm Y_lm with c_lm ~ N(0, 0.1 / l), l <= min(16, nt / 4), and a
    density band around the equator with noise."""
    rng = np.random.default_rng(seed)
    h, L = math.pi / nt, max(1, min(16, nt // 4))
    theta = np.arange(nt + 1) * h
    x, s = np.cos(theta), np.sin(theta)
    A, B = np.zeros((nt + 1, L + 1)), np.zeros((nt + 1, L + 1))
    pmm = np.full(nt + 1, math.sqrt(0.25 / math.pi))
    for m in range(L + 1):  # normalised associated Legendre functions, upwards in l
        if m:
            pmm = pmm * s * math.sqrt((2 * m + 1) / (2 * m))
        p0, p1 = np.zeros(nt + 1), pmm
        for l in range(m, L + 1):
            if l > m:
                a = math.sqrt((4 * l * l - 1) / (l * l - m * m))
                b = math.sqrt(((l - 1) ** 2 - m * m) / (4 * (l - 1) ** 2 - 1))
                p0, p1 = p1, a * (x * p1 - b * p0)
            if l:
                A[:, m] += 0.1 / l * rng.standard_normal() * p1 * (math.sqrt(2) if m else 1.0)
                B[:, m] += 0.1 / l * rng.standard_normal() * p1 * (math.sqrt(2) if m else 0.0)
    phi = (np.arange(2 * nt) - 0.5) * h
    m = np.arange(L + 1)[:, None]
    psi = A @ np.cos(m * phi) + B @ np.sin(m * phi)
    u_phi = (psi[1:] - psi[:-1]) / h
    u_theta = -(np.roll(psi, -1, axis=1) - psi)[1:-1] / (h * s[1:-1, None])
    band = np.clip(0.5 + (0.3 - np.abs((np.arange(nt) + 0.5) * h - 0.5 * math.pi)) / (2 * h), 0.0, 1.0)
    rho = 0.8 * band[:, None] + 0.1 * rng.random((nt, 2 * nt))
    return [np.ascontiguousarray(a, np.float32) for a in (u_phi, u_theta, rho)]


def _particles(n, seed):
    """n particles (phi, theta) spread over the sphere."""
    rng = np.random.default_rng(seed + 77)
    phi = 2 * math.pi * rng.random(n)
    return np.stack([phi, np.arccos(1 - 2 * (1e-4 + 0.9998 * rng.random(n)))], axis=1).astype(np.float32)


class _Noalloc:
    def __init__(self, case, seed):
        nt = case["nt"]
        u_phi, u_theta, rho = (torch.from_numpy(a).cuda() for a in _fields(nt, seed))
        self.fields = [u_phi, u_theta] + ([rho] if case["density"] else [])
        self.desc = K.SimDesc(nt, 2 * nt, 1.0, 0.5 / nt, int(case["geometric"]), int(case["fp64"]), 0)
        self.step = K.lib().kam_sim_step_noalloc
        self.steps = case["steps"]

    def run(self):
        p = [f.data_ptr() for f in self.fields] + [None]
        K.check(self.step(C.byref(self.desc), p[0], p[1], p[2], self.steps, torch.cuda.current_stream().cuda_stream))
        return self.fields


class _Frame:
    def __init__(self, case, seed):
        nt = case["nt"]
        self.sim = K.Sim(nt, 0.5 / nt, precision=int(case["fp64"]))
        self.sim.set_fields(*_fields(nt, seed))
        self.particles = case["particles"] > 0
        if self.particles:
            self.sim.set_particles(_particles(case["particles"], seed))
        self.steps = case["steps"]

    def run(self):
        self.sim.step(self.steps)
        out = list(self.sim.get_fields())
        return out + [self.sim.get_particles()] if self.particles else out


class _Engine:
    """The engine with its residents, and the requests that come and go in each pass."""

    def __init__(self, case, seed):
        self.requests, residents = _members(case)
        self.precision, self.graph = int(case["fp64"]), case["graph"]
        total = sum(K.lib().kam_sim_bytes(n, 2 * n) + 4096 for n in residents + [r[0] for r in self.requests])
        self.eng = K.Engine(hbm_budget_bytes=total + (64 << 20), use_graph=self.graph,
                            graph_steps=32 if self.graph else 1, groups=3)
        variants = {}
        for k, nt in enumerate(residents):
            key = (nt, k % 4)
            if key not in variants:
                variants[key] = _fields(nt, 1000 + 17 * seed + k % 4)
            if self.eng.admit(nt, 0.5 / nt, *variants[key], steps=10 ** 9, precision=self.precision) is None:
                raise RuntimeError("the engine refused a resident")
        self.inputs = [_fields(nt, 100 * seed + k) for k, (nt, _) in enumerate(self.requests)]
        self.eng.step(1)
        self.eng.sync()

    def run(self):
        eng, ids = self.eng, []
        for (nt, steps), fields in zip(self.requests, self.inputs):
            ids.append(eng.admit(nt, 0.5 / nt, *fields, steps=steps, precision=self.precision))
        eng.step(max(steps for _, steps in self.requests))
        return [eng.fetch(rid, nt) for rid, (nt, _) in zip(ids, self.requests)]


def prepare(case, seed):
    return {"noalloc": _Noalloc, "frame": _Frame, "engine": _Engine}[case["entry"]](case, seed)


def run(state):
    return state.run()


def work(case):
    """Each field read once and written once in the pass (4 bytes a value), particles likewise; and the floating-point
    operations of the steps: per cell 9 bilinear samples (9 each), the departure points and averages (40), the metric
    update (25), divergence and gradient (14), the tridiagonal solve (20) and two real FFTs (2.5 log2 n_phi each)."""
    if case["entry"] == "engine":
        requests, residents = _members(case)
        most = max(s for _, s in requests)
        spheres = [(nt, s) for nt, s in requests] + [(nt, most) for nt in residents]
    else:
        spheres = [(case["nt"], case["steps"])]
    b = sum(24 * 2 * nt * nt for nt, _ in spheres)
    f = sum(s * 2 * nt * nt * (180 + 5 * math.log2(2 * nt)) for nt, s in spheres)
    if case["entry"] == "frame":
        b += 16 * case["particles"]
        f += 50 * case["particles"] * case["steps"]
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# The step in 64 bits, in torch
# ---------------------------------------------------------------------------
# offsets of the u_phi, u_theta and centred grids in cells
_OFF = [(-0.5, 0.5), (0.0, 1.0), (0.0, 0.5)]


def _sample(kind, f, phi, theta):
    """Bilinear sample of grid `kind` at (phi, theta) in cells, folded over the poles."""
    rows, n_phi = f.shape
    nt = n_phi // 2
    p, t = phi - _OFF[kind][0], theta - _OFF[kind][1]
    t = t - torch.floor(t / n_phi) * n_phi
    flip = t > nt
    t = torch.where(flip, n_phi - t, t)
    p = torch.where(flip, p + nt, p)
    p = p - torch.floor(p / n_phi) * n_phi
    ip, it = torch.floor(p), torch.floor(t)
    ap, at = p - ip, t - it
    i0, j = ip.long() % n_phi, it.long()
    pole = ((j == 0) & flip) | (j == (nt - 2 if kind == 1 else nt - 1))
    r0 = j.clamp(0, rows - 1)
    r1 = torch.where(pole, r0, (j + 1).clamp(0, rows - 1))
    k0 = torch.where(pole, (i0 + nt) % n_phi, i0)
    at = torch.where(pole, at if kind == 0 else 0.5 * at, at)
    g = f.reshape(-1)
    lo = (1 - ap) * g[r0 * n_phi + i0] + ap * g[r0 * n_phi + (i0 + 1) % n_phi]
    hi = (1 - ap) * g[r1 * n_phi + k0] + ap * g[r1 * n_phi + (k0 + 1) % n_phi]
    return (1 - at) * lo + at * hi


def _advect(kind, src, u_phi, u_theta, dt):
    rows, n_phi = src.shape
    h = 2 * math.pi / n_phi
    opt = dict(dtype=src.dtype, device=src.device)
    gp = (torch.arange(n_phi, **opt) + _OFF[kind][0])[None, :].expand(rows, n_phi)
    gt = (torch.arange(rows, **opt) + _OFF[kind][1])[:, None].expand(rows, n_phi)
    cp, ct = dt / (h * torch.sin(gt * h)), dt / h
    up, ut = _sample(0, u_phi, gp, gt), _sample(1, u_theta, gp, gt)
    mp, mt = gp - 0.5 * cp * up, gt - 0.5 * ct * ut
    vp, vt = _sample(0, u_phi, mp, mt), _sample(1, u_theta, mp, mt)
    return _sample(kind, src, gp - 0.5 * cp * (up + vp), gt - 0.5 * ct * (ut + vt))


def _metric(u_phi, u_theta, dt):
    """The root x of G^2 x^3 + (1 + G v) x - u = 0 and v + G x^2 per cell, taken back to the staggered grids."""
    nt, n_phi = u_phi.shape
    th = (torch.arange(nt, dtype=u_phi.dtype, device=u_phi.device)[:, None] + 0.5) * (math.pi / nt)
    u = 0.5 * (u_phi + torch.roll(u_phi, -1, 1))
    v = torch.empty_like(u_phi)
    v[1:-1] = 0.5 * (u_theta[:-1] + u_theta[1:])
    for row in (0, -1):
        v[row] = 0.75 * u_theta[row] + 0.25 * torch.roll(u_theta[row], -nt)
    G = dt * torch.cos(th) / torch.sin(th)
    a, b = G * G, 1 + G * v
    up = b > 0  # one real root: Newton from the smaller of its two bounds
    bs = torch.where(up, b, torch.ones_like(b))
    x = torch.minimum(u.abs() / bs, (u.abs() / torch.where(a > 0, a, 1e-300 + 0 * a)) ** (1 / 3))
    for _ in range(50):
        x = x - (a * x ** 3 + bs * x - u.abs()) / (3 * a * x * x + bs)
    x = torch.copysign(x, u)
    if not bool(up.all()):  # three real roots possible: the one Cardano's formula gives
        q, r = -b / (3 * a), -u / (2 * a)
        trig = r * r <= q ** 3 + 1e-7
        y = -2 * torch.sqrt(q.clamp(min=0)) * torch.cos(torch.acos((r / q.clamp(min=1e-300) ** 1.5).clamp(-1, 1)) / 3)
        c = -torch.copysign((r.abs() + torch.sqrt((r * r - q ** 3).clamp(min=0))) ** (1 / 3), r)
        x = torch.where(up, x, torch.where(trig, y, c + q / c))
    x = torch.where(G.abs() > 1e-7, x, u)
    w = v + G * x * x
    return 0.5 * (x + torch.roll(x, 1, 1)), 0.5 * (w[:-1] + w[1:])


def _project(u_phi, u_theta):
    nt, n_phi = u_phi.shape
    h = math.pi / nt
    opt = dict(dtype=u_phi.dtype, device=u_phi.device)
    tc = (torch.arange(nt, **opt)[:, None] + 0.5) * h
    flux = torch.zeros(nt + 1, n_phi, **opt)
    flux[1:-1] = u_theta * torch.sin((torch.arange(1, nt, **opt) * h))[:, None]
    d = (flux[1:] - flux[:-1] + torch.roll(u_phi, -1, 1) - u_phi) / (h * torch.sin(tc))
    dh = torch.fft.rfft(d, dim=1)[:, 1:].T.contiguous()  # [mode 1 .. n_phi/2][row]
    n = torch.arange(1, nt + 1, **opt)[:, None]
    s, ct = torch.sin(tc).T, (torch.cos(tc) / torch.sin(tc)).T / (2 * h)
    a, c = (1 / h ** 2 - ct).expand(nt, nt).clone(), (1 / h ** 2 + ct).expand(nt, nt).clone()
    b = -2 / h ** 2 - n * n / (s * s)
    b[:, 0] += a[:, 0]
    b[:, -1] += c[:, -1]
    a[:, 0] = 0
    c[:, -1] = 0
    st = 1
    while st < nt:  # parallel cyclic reduction
        def at(x, k, fill=0.0):
            y = torch.full_like(x, fill)
            if k > 0:
                y[:, k:] = x[:, :-k]
            else:
                y[:, :k] = x[:, -k:]
            return y
        k1, k2 = a / at(b, st, 1.0), c / at(b, -st, 1.0)
        b, dh = b - at(c, st) * k1 - at(a, -st) * k2, dh - at(dh, st) * k1 - at(dh, -st) * k2
        a, c = -at(a, st) * k1, -at(c, -st) * k2
        st *= 2
    ph = torch.zeros(nt, nt + 1, dtype=dh.dtype, device=dh.device)
    ph[:, 1:] = (dh / b).T
    p = torch.fft.irfft(ph, n=n_phi, dim=1)
    return u_phi - (p - torch.roll(p, 1, 1)) / (h * torch.sin(tc)), u_theta - (p[1:] - p[:-1]) / h


def _steps(nt, fields, steps, geometric=True, particles=None):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    up, ut, rho = (torch.from_numpy(f).to(dev, torch.float64) for f in fields)
    if particles is not None:
        particles = torch.from_numpy(particles).to(dev, torch.float64)
    dt, h = 0.5 / nt, math.pi / nt
    for _ in range(steps):
        if particles is not None:
            ph, th = particles[:, 0], particles[:, 1]
            vp, vt = _sample(0, up, ph / h, th / h), _sample(1, ut, ph / h, th / h)
            ph, th = ph + dt * vp / torch.sin(th), th + dt * vt
            over = (th < 0) | (th > math.pi)
            th = torch.where(th < 0, -th, torch.where(th > math.pi, 2 * math.pi - th, th))
            particles = torch.stack([torch.remainder(torch.where(over, ph + math.pi, ph), 2 * math.pi), th], dim=1)
        a, b, rho = _advect(0, up, up, ut, dt), _advect(1, ut, up, ut, dt), _advect(2, rho, up, ut, dt)
        if geometric:
            a, b = _metric(a, b, dt)
        up, ut = _project(a, b)
    return [up, ut, rho] + ([] if particles is None else [particles])


def exact(case, seed):
    if case["entry"] == "engine":
        requests, _ = _members(case)
        if sum(nt * nt * s for nt, s in requests) > 1.2e8:
            return None
        return [tuple(_steps(nt, _fields(nt, 100 * seed + k), s)) for k, (nt, s) in enumerate(requests)]
    nt = case["nt"]
    if nt * nt * case["steps"] > 1.2e8:
        return None
    if case["entry"] == "frame":
        return _steps(nt, _fields(nt, seed), case["steps"],
                      particles=_particles(case["particles"], seed) if case["particles"] else None)
    fields = _fields(nt, seed)
    out = _steps(nt, fields, case["steps"], geometric=case["geometric"])
    return out if case["density"] else out[:2]
