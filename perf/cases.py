"""Timed workloads of the el_iso RK4 time-stepping path.

A case is one model with its resident session(s) and one pass is what a
modelling program does with it again and again: advance every shot by a chunk
of time steps, read the seismograms of the chunk, and read the snapshot planes
(the surface and a vertical section; for shots from rest, the two planes
through the source) that such a program writes after it.  Sessions, model
uploads and initial fields are made once, as a program would.

`exact` is the same scheme in 64 bits, written with torch from the equations:
MacCormack/DRP differences in curvilinear coordinates, the traction image and
the velocity conversion on a free surface, CFS-PML memory variables, classical
RK4, point sources and trilinear receivers.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "gpu-cgfd3d-elastic_amd"))

import cgfd  # noqa: E402

NG = 3
H = 100.0      # grid spacing, m
DT = 0.005     # time step, s
VX, VY, VZ, TXX, TYY, TZZ, TYZ, TXZ, TXY = range(9)
STORES = {"f32": (cgfd.STORE_F32, 4, 4), "f16": (cgfd.STORE_F16, 2, 4), "bf16": (cgfd.STORE_BF16, 2, 4),
          "f64": (cgfd.STORE_F64, 8, 8)}


def _case(name, ni, nj, nk, grid, storage, shots, steps, top="free", nlay=10, start="restart", nrecv=20,
          source="moment", peak=False):
    return dict(name=name, ni=ni, nj=nj, nk=nk, grid=grid, storage=storage, shots=shots, steps=steps, top=top,
                nlay=nlay, start=start, nrecv=nrecv, source=source, peak=peak)


def listed():
    return [
        # the smallest model a server keeps resident: launch latency decides
        _case("topo-64-f32", 64, 64, 64, "topography", "f32", 1, 32),
        # a double-precision check of a small sheared grid with odd extents
        _case("curv-67x53x45-f64", 67, 53, 45, "curvilinear", "f64", 1, 16, nlay=6, nrecv=6, source="force"),
        # one shot on the 100x100x60 explosion model
        _case("explosion-100-f32", 100, 100, 60, "cartesian", "f32", 1, 40),
        # the same medium serving batches of shots, each from rest
        _case("explosion-100-batch64-f32", 100, 100, 60, "cartesian", "f32", 64, 24, start="rest"),
        _case("explosion-100-batch16-f16", 100, 100, 60, "cartesian", "f16", 16, 32),
        # ordinary regional models with topography, single and half storage
        _case("topo-256-f32", 256, 256, 128, "topography", "f32", 1, 24, nrecv=400),
        _case("topo-211x187x121-bf16", 211, 187, 121, "topography", "bf16", 1, 21, nrecv=400),
        # a grid sheared in every direction, with the surface's peak motion
        _case("curv-200x180x100-f32", 200, 180, 100, "curvilinear", "f32", 1, 24, nrecv=100, peak=True),
        # a buried full-space model: absorbing layers on all six faces
        _case("fullspace-173x129x97-f32", 173, 129, 97, "cartesian", "f32", 1, 19, top="pml", nlay=12,
              source="force"),
        # the double-precision reference path on an ordinary model
        _case("topo-128x128x96-f64", 128, 128, 96, "topography", "f64", 1, 24),
        # large models from rest, single and half storage
        _case("explosion-400-f32", 400, 400, 200, "cartesian", "f32", 1, 24, start="rest"),
        _case("explosion-400-f16", 400, 400, 200, "cartesian", "f16", 1, 24, start="rest"),
    ]


def draw(rng):
    points = math.exp(rng.uniform(math.log(6e4), math.log(1.4e7)))
    nk = max(36, int(round((points * rng.uniform(0.15, 0.8)) ** (1 / 3))))
    ar = math.exp(rng.uniform(math.log(0.6), math.log(1.6)))
    ni = max(36, int(round(math.sqrt(points / nk * ar))))
    nj = max(36, int(round(math.sqrt(points / nk / ar))))
    n = ni * nj * nk
    shots = rng.choice([1, 1, 1, 2, 5, 16, 64])
    shots = max(1, min(shots, int(3e7 / n)))
    total = n * shots
    storage = rng.choice(["f32", "f32", "f32", "f16", "f16", "bf16", "f64"])
    steps = rng.randint(8, 33) if total < 8e6 else rng.randint(8, 24)
    return _case("", ni, nj, nk, rng.choice(["cartesian", "topography", "topography", "curvilinear"]), storage, shots,
                 steps, top=rng.choice(["free", "free", "free", "pml"]), nlay=rng.choice([6, 8, 10, 12]),
                 start="restart" if total < 8e6 else "rest", nrecv=rng.choice([5, 20, 100]),
                 source=rng.choice(["moment", "moment", "force"]), peak=rng.random() < 0.2)


# ------------------------------------------------------------------ model
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _coords(case, rng):
    """The nine first derivatives of (x, y, z) on every point, ghosts included:
    [3][3][nz][ny][nx] as d(x, y, z) / d(i, j, k)."""
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    dev = _device()
    t = dict(dtype=torch.float64, device=dev)
    i = (torch.arange(ni + 2 * NG, **t) - NG)[None, None, :]
    j = (torch.arange(nj + 2 * NG, **t) - NG)[None, :, None]
    k = (torch.arange(nk + 2 * NG, **t) - NG)[:, None, None]
    shape = (nk + 2 * NG, nj + 2 * NG, ni + 2 * NG)
    zero = torch.zeros(shape, **t)
    d = [[zero.clone() for _ in range(3)] for _ in range(3)]
    d[0][0] += H
    d[1][1] += H
    if case["grid"] == "cartesian":
        d[2][2] += H
        return d
    # surface: three hills and a short-wavelength roughness that fade with
    # depth; vertical spacing grows from H at the top to 1.5 H at the bottom
    surf, s_i, s_j = 0.0, 0.0, 0.0
    for _ in range(3):
        amp = rng.uniform(300.0, 800.0) * min(1.0, nk / 200.0)
        sig = rng.uniform(0.12, 0.3) * min(ni, nj) * H
        ci, cj = rng.uniform(0.2, 0.8) * ni, rng.uniform(0.2, 0.8) * nj
        g = amp * torch.exp(-(((i - ci) * H) ** 2 + ((j - cj) * H) ** 2) / (2 * sig ** 2))
        surf, s_i, s_j = surf + g, s_i - g * (i - ci) * H * H / sig ** 2, s_j - g * (j - cj) * H * H / sig ** 2
    for _ in range(4):
        ki, kj, ph = rng.uniform(-0.3, 0.3), rng.uniform(-0.3, 0.3), rng.uniform(0, 2 * math.pi)
        c = 25.0 * torch.cos(ki * i + kj * j + ph)
        s = 25.0 * torch.sin(ki * i + kj * j + ph)
        surf, s_i, s_j = surf + c, s_i - ki * s, s_j - kj * s
    u = (nk - 1 - k) / (nk - 1)
    d[2][0] += (1 - u) * s_i
    d[2][1] += (1 - u) * s_j
    d[2][2] += surf / (nk - 1) + H * (1 + 0.5 * u)
    if case["grid"] == "curvilinear":
        p, q = rng.uniform(0.08, 0.2), rng.uniform(0.08, 0.2)
        a = 0.4 * H
        d[0][1] += a * p * torch.cos(p * j)
        d[0][2] += a * q * torch.cos(q * k)
        d[1][0] -= a * q * torch.sin(q * i)
        d[1][2] -= a * p * torch.sin(p * k)
    return d


def _metric(d):
    """[10][nz][ny][nx]: the Jacobian and the rows grad xi, grad eta, grad zeta."""
    cof = [[d[(c + 1) % 3][(r + 1) % 3] * d[(c + 2) % 3][(r + 2) % 3]
            - d[(c + 1) % 3][(r + 2) % 3] * d[(c + 2) % 3][(r + 1) % 3] for c in range(3)] for r in range(3)]
    jac = d[0][0] * cof[0][0] + d[1][0] * cof[0][1] + d[2][0] * cof[0][2]
    return torch.stack([jac] + [cof[r][c] / jac for r in range(3) for c in range(3)])


def _medium(case, rng, shape):
    """lam, mu, 1/rho."""
    t = dict(dtype=torch.float64, device=_device())
    nz, ny, nx = shape
    if case["grid"] == "cartesian":
        vp, vs, rho = (torch.full(shape, v, **t) for v in (6000.0, 3464.0, 2670.0))
    else:
        i = torch.arange(nx, **t)[None, None, :]
        j = torch.arange(ny, **t)[None, :, None]
        k = torch.arange(nz, **t)[:, None, None]
        vp = torch.full(shape, 6500.0, **t)
        vp = torch.where(k > 0.45 * nz, torch.full_like(vp, 5000.0), vp)
        vp = torch.where(k > 0.8 * nz, torch.full_like(vp, 3000.0), vp)
        for _ in range(4):
            w = [rng.uniform(-0.5, 0.5) for _ in range(3)]
            vp = vp * (1 + 0.012 * torch.sin(w[0] * i + w[1] * j + w[2] * k + rng.uniform(0, 6.28)))
        vs, rho = vp / 1.73, 310.0 * vp ** 0.25
    mu = rho * vs * vs
    return rho * vp * vp - 2 * mu, mu, 1.0 / rho


def _surface_matrices(metric, lam, mu, nk):
    """dV/dzeta of a traction-free surface from dV/dxi and dV/deta, [ny][nx][9] each."""
    k = NG + nk - 1
    e = metric[1:, k].reshape(3, 3, *metric.shape[2:])
    lm, m = lam[k][..., None, None], mu[k][..., None, None]
    n = e[2].permute(1, 2, 0)
    eye = torch.eye(3, dtype=metric.dtype, device=metric.device)

    def op(v):
        v = v.permute(1, 2, 0)
        return (lm * n[..., :, None] * v[..., None, :] + m * v[..., :, None] * n[..., None, :]
                + m * (n * v).sum(-1)[..., None, None] * eye)

    a = op(e[2])
    return [torch.linalg.solve(a, -op(e[r])).reshape(*a.shape[:2], 9) for r in (0, 1)]


def _profile(nlay, face):
    """CFS-PML A, B, D along one face, low index to high."""
    length = nlay * H
    refl = 10.0 ** -((math.log10(nlay) - 1.0) / math.log10(2.0) + 4.0)
    d0 = -6000.0 / (2.0 * length) * math.log(refl) * 3.0
    n = np.arange(nlay + 1)
    r = n / nlay
    d, a, b = d0 * r * r, 3.0 * (1 - r), 1.0 + 1.5 * r * r
    abd = [a + d / b, 1.0 / b, d / b]
    return [v[::-1].copy() if face % 2 == 0 else v for v in abd]


def _field(case, rng):
    """A developed wavefield, smooth and fading towards the sides: [9][nz][ny][nx], ghosts zero."""
    ni, nj, nk, nlay = case["ni"], case["nj"], case["nk"], case["nlay"]
    t = dict(dtype=torch.float64, device=_device())
    i = torch.arange(ni, **t)[None, None, :]
    j = torch.arange(nj, **t)[None, :, None]
    k = torch.arange(nk, **t)[:, None, None]

    def fade(x, n):
        return torch.sin(torch.clamp((x + 1) / (nlay + 4.0), max=1.0) * math.pi / 2) ** 2

    win = fade(i, ni) * fade(ni - 1 - i, ni) * fade(j, nj) * fade(nj - 1 - j, nj) * fade(k, nk)
    if case["top"] == "pml":
        win = win * fade(nk - 1 - k, nk)
    w = torch.zeros((9, nk + 2 * NG, nj + 2 * NG, ni + 2 * NG), **t)
    for c in range(9):
        v = 0.0
        for _ in range(4):
            a, p = rng.uniform(0.1, 0.25), rng.uniform(0, 6.28)
            v = v + a * torch.sin(rng.uniform(-0.6, 0.6) * i + rng.uniform(-0.6, 0.6) * j
                                  + rng.uniform(-0.6, 0.6) * k + p)
        w[c, NG:NG + nk, NG:NG + nj, NG:NG + ni] = v * win * (1.0 if c < 3 else 8e6)
    return w


def _source(case, rng):
    """One point source: Ricker time function at the four stage times, 7x7x7 Gaussian weights."""
    ni, nj, nk, steps, lay = case["ni"], case["nj"], case["nk"], case["steps"], case["nlay"] + 1
    ci, cj = rng.randint(lay + 4, ni - lay - 5), rng.randint(lay + 4, nj - lay - 5)
    ck = rng.randint(lay + 4, nk - 10 if case["top"] == "free" else nk - lay - 5)
    f0, t0 = rng.uniform(2.0, 8.0), rng.uniform(0.3, 0.6) * steps * DT
    it = np.arange(steps)[:, None] * DT + np.array([0.0, 0.5, 0.5, 1.0])[None, :] * DT - t0
    u = (math.pi * f0 * it) ** 2
    stf = (1 - 2 * u) * np.exp(-u)
    o = np.arange(-3, 4)
    dk, dj, di = (g.ravel() for g in np.meshgrid(o, o, o, indexing="ij"))
    wgt = np.exp(-(di ** 2 + dj ** 2 + dk ** 2) / 4.0)
    idx = ((ck + dk + NG) * (nj + 2 * NG) + (cj + dj + NG)) * (ni + 2 * NG) + ci + di + NG
    if case["source"] == "moment":
        mom = [rng.gauss(0.0, 1.0) * 1e16 for _ in range(6)]
        F, M = None, np.stack([stf * m for m in mom]).reshape(6, 1, steps, 4)
    else:
        frc = [rng.gauss(0.0, 1.0) * 1e12 for _ in range(3)]
        F, M = np.stack([stf * f for f in frc]).reshape(3, 1, steps, 4), None
    return dict(nsrc=1, force_on=int(F is not None), moment_on=int(M is not None), max_nt=steps, max_ext=343,
                it_begin=np.array([0]), it_end=np.array([steps - 1]), ext_num=np.array([343]),
                ext_indx=idx, ext_coef=wgt / wgt.sum(), F=F, M=M), (ci, cj, ck)


def _receivers(case, rng, at):
    """Half on the surface plane, half around the source; every other one between nodes in x and y."""
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    ny, nx = nj + 2 * NG, ni + 2 * NG
    idx, frac = [], []
    for r in range(case["nrecv"]):
        if r % 2 == 0 and case["top"] == "free":
            i, j, k = rng.randrange(ni - 1), rng.randrange(nj - 1), nk - 1
        else:
            i, j, k = (max(0, min(n - 2, c + rng.randint(-8, 8))) for c, n in zip(at, (ni, nj, nk)))
        p = ((k + NG) * ny + j + NG) * nx + i + NG
        idx.append([p + a + b * nx + c * nx * ny for c in (0, 1) for b in (0, 1) for a in (0, 1)])
        frac.append([0.0, 0.0, 0.0] if r % 2 else [rng.random() * 0.9, rng.random() * 0.9, 0.0])
    return np.array(idx), np.array(frac)


def _inputs(case, seed):
    """Everything a pass is given, as the arrays the session receives (in its model type)."""
    import random
    rng = random.Random(int(seed) * 7919 + 17)
    f = np.float64 if case["storage"] == "f64" else np.float32

    def host(v):
        return v.to(torch.float64 if f is np.float64 else torch.float32).cpu().numpy()

    def cast(src):
        return {k: (np.asarray(v, f) if k in ("ext_coef", "F", "M") and v is not None else v)
                for k, v in src.items()}

    metric = _metric(_coords(case, rng))
    lam, mu, slw = _medium(case, rng, metric.shape[1:])
    m = dict(metric=host(metric), lam=host(lam), mu=host(mu), slw=host(slw))
    if case["top"] == "free":
        m["mvx"], m["mvy"] = (host(v) for v in _surface_matrices(metric, lam, mu, case["nk"]))
    faces = range(5 if case["top"] == "free" else 6)
    m["pml"] = {p: [np.asarray(v, f) for v in _profile(case["nlay"], p)] for p in faces}
    m["shots"] = []
    for _ in range(case["shots"]):
        src, at = _source(case, rng)
        idx, frac = _receivers(case, rng, at)
        m["shots"].append(dict(src=cast(src), idx=idx, frac=np.asarray(frac, f), planes=_planes(case, at),
                               w=host(_field(case, rng)) if case["start"] == "restart" else None))
    return m


def prepare(case, seed):
    m = _inputs(case, seed)
    s = cgfd.Session(case["ni"], case["nj"], case["nk"], storage=STORES[case["storage"]][0], nshots=case["shots"])
    s.upload_metric(m["metric"])
    s.upload_medium(m["lam"], m["mu"], m["slw"])
    if case["top"] == "free":
        s.upload_free_surface(True, m["mvx"], m["mvy"])
    else:
        s.upload_free_surface(False)
    for face, (a, b, d) in m["pml"].items():
        s.upload_pml(face, case["nlay"], a, b, d)
    if STORES[case["storage"]][1] == 2:
        s.set_storage_scale([-3] * 3 + [20] * 6)
    if case["peak"] and case["top"] == "free":
        s.set_peak_motion(True)
    for n, shot in enumerate(m["shots"]):
        if shot["w"] is not None:
            s.set_level(n, cgfd.LEVEL_PRE, shot["w"])
        s.upload_source(n, shot["src"])
        s.upload_receivers(n, shot["idx"], shot["frac"], case["steps"])
    return dict(case=case, session=s, planes=[shot["planes"] for shot in m["shots"]])


def _snapshot_shots(case):
    return range(min(case["shots"], 2))


def _planes(case, at):
    """(j, k) of the vertical and the horizontal plane a shot's snapshots hold."""
    return (at[1], at[2]) if case["start"] == "rest" else (case["nj"] // 2, case["nk"] - 1)


def run(state):
    case, s = state["case"], state["session"]
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    t = np.float64 if case["storage"] == "f64" else np.float32
    s.run(0, case["steps"], DT)
    out = {"seismograms": np.stack([s.read_seismo(n, t) for n in range(case["shots"])])}
    for n in _snapshot_shots(case):
        j, k = state["planes"][n]
        out["plane%d" % n] = s.fetch_subvolume(n, cgfd.LEVEL_PRE, range(9), (0, 0, k), (ni, nj, 1), dtype=t)
        out["section%d" % n] = s.fetch_subvolume(n, cgfd.LEVEL_PRE, range(9), (0, j, 0), (ni, 1, nk), dtype=t)
    if case["peak"] and case["top"] == "free":
        out["peak"] = s.read_peak_motion(0, t)
    return out


def work(case):
    """RK4 with a right-hand side at each stage: each stage reads its input and the coefficients once and writes
    its output once, W^n is read by the three later stages, and the last one takes two of the stage values
    (or their sum) besides: 117 wavefield words per point and step.  A Cartesian grid has 3 coefficients per
    point (lam, mu, 1/rho), a grid of vertical lines 3 more, a general one 12.  The memory variables of a
    point in an absorbing layer follow the wavefield."""
    n, shots = case["ni"] * case["nj"] * case["nk"], case["shots"]
    _, ws, ms = STORES[case["storage"]]
    lay = case["nlay"] + 1
    pairs = 2 * lay * (case["nj"] * case["nk"] + case["ni"] * case["nk"])
    pairs += (1 if case["top"] == "free" else 2) * lay * case["ni"] * case["nj"]
    coef = {"cartesian": 3, "topography": 6, "curvilinear": 12}[case["grid"]]
    step = shots * ((n + pairs) * 117 * ws) + 4 * n * coef * ms
    return {"bytes": float(case["steps"] * step), "flops": float(case["steps"] * shots * n * 4 * 430)}


# ------------------------------------------------------------------ the scheme in 64 bits
COEF = {0: (-3, (-0.041686285, 0.333411808, -1.250117713, 0.666745142, 0.291647047)),
        1: (-1, (-0.291647047, -0.666745142, 1.250117713, -0.333411808, 0.041686285))}
PAIRS = [(0, 0, 0), (1, 1, 0), (1, 1, 1), (0, 0, 1), (0, 1, 0), (1, 0, 0), (1, 0, 1), (0, 1, 1)]
STRESS = ((TXX, TXY, TXZ), (TXY, TYY, TYZ), (TXZ, TYZ, TZZ))


class _Scheme:
    def __init__(self, case, m):
        dev = _device()
        self.c, self.n = case, (case["nk"], case["nj"], case["ni"])
        nk, nj, ni = self.n
        t = lambda v: torch.from_numpy(np.asarray(v, np.float64)).to(dev)  # noqa: E731
        self.met = t(m["metric"])
        self.inner = tuple(slice(NG, NG + v) for v in self.n)
        phys = lambda v: v[self.inner]  # noqa: E731
        self.e = [[phys(self.met[1 + 3 * r + c]) for c in range(3)] for r in range(3)]
        self.jac = phys(self.met[0])
        self.lam, self.mu, self.slw = (phys(t(m[q])) for q in ("lam", "mu", "slw"))
        self.free = case["top"] == "free"
        if self.free:
            self.mats = [t(m[q])[NG:NG + nj, NG:NG + ni].permute(2, 0, 1).reshape(3, 3, nj, ni) for q in ("mvx", "mvy")]
        lay = case["nlay"] + 1
        self.faces = []
        for p, abd in m["pml"].items():
            ax = 2 - p // 2
            box = [slice(0, v) for v in self.n]
            box[ax] = slice(0, lay) if p % 2 == 0 else slice(self.n[ax] - lay, self.n[ax])
            form = [1, 1, 1]
            form[ax] = lay
            self.faces.append((p // 2, tuple(box), [t(v).reshape(form) for v in abd]))

    def diff(self, f, axis, way):
        lo, co = COEF[way]
        out = 0.0
        for q, c in enumerate(co):
            s = list(self.inner)
            s[axis] = slice(NG + lo + q, NG + lo + q + self.n[axis])
            out = out + c * f[tuple(s)]
        return out

    def hooke(self, g):
        """Stress rates of a velocity gradient g[a][b] = dV_a/dx_b."""
        return self._hooke(g, self.lam, self.mu)

    @staticmethod
    def _hooke(g, lam, mu):
        tr = lam * (g[0][0] + g[1][1] + g[2][2])
        return {TXX: tr + 2 * mu * g[0][0], TYY: tr + 2 * mu * g[1][1], TZZ: tr + 2 * mu * g[2][2],
                TXY: mu * (g[0][1] + g[1][0]), TXZ: mu * (g[0][2] + g[2][0]), TYZ: mu * (g[1][2] + g[2][1])}

    def image(self, w, ways, h):
        """Momentum rows next to the surface: conservative form, odd image of the traction."""
        nk = self.n[0]
        top, lo_row = nk - 1, nk - 5
        rows = slice(NG + lo_row, NG + nk)
        met = self.met[:, rows]
        first = top - (1 if ways[2] == 0 else 3)
        keep = slice(first - lo_row, 5)
        jn, in_ = self.inner[1], self.inner[2]
        for a in range(3):
            vec = [met[0] * sum(met[1 + 3 * r + b] * w[STRESS[a][b]][rows] for b in range(3)) for r in range(3)]
            tot = 0.0
            for r, axis in ((0, 2), (1, 1)):
                lo, co = COEF[ways[r]]
                for q, c in enumerate(co):
                    s = [keep, jn, in_]
                    s[axis] = slice(NG + lo + q, NG + lo + q + self.n[axis])
                    tot = tot + c * vec[r][tuple(s)]
            z = vec[2][:, jn, in_]
            z = torch.cat([z[:4], torch.zeros_like(z[:1]), -z[3:4], -z[2:3], -z[1:2]])
            lo, co = COEF[ways[2]]
            for q, c in enumerate(co):
                tot = tot + c * z[first - lo_row + lo + q:5 + lo + q]
            h[a][first:] = tot * self.slw[first:] / self.jac[first:]

    def rhs(self, w, aux, ways):
        """Rates of the wavefield (physical points) and of each face's memory variables."""
        axes = (2, 1, 0)
        D = [[self.diff(w[c], axes[r], ways[r]) for c in range(9)] for r in range(3)]
        e, nk = self.e, self.n[0]
        h = [None] * 9
        for a in range(3):
            h[a] = self.slw * sum(e[r][b] * D[r][STRESS[a][b]] for r in range(3) for b in range(3))
        dz = [D[2][a] for a in range(3)]
        if self.free:
            self.image(w, ways, h)
            dz = [v.clone() for v in dz]
            wi = [w[a][:, self.inner[1], self.inner[2]] for a in range(3)]
            row = lambda a, k: wi[a][NG + k]  # noqa: E731
            for a in range(3):
                dz[a][nk - 1] = sum(self.mats[r][a, b] * D[r][b][nk - 1] for r in (0, 1) for b in range(3))
                k = nk - 2
                dz[a][k] = row(a, k) - row(a, k - 1) if ways[2] == 0 else row(a, k + 1) - row(a, k)
                k = nk - 3
                dz[a][k] = ((row(a, k - 2) - 8 * row(a, k - 1) + 7 * row(a, k)) / 6 if ways[2] == 0
                            else (-7 * row(a, k) + 8 * row(a, k + 1) - row(a, k + 2)) / 6)
        g = [[e[0][b] * D[0][a] + e[1][b] * D[1][a] + e[2][b] * dz[a] for b in range(3)] for a in range(3)]
        for c, v in self.hooke(g).items():
            h[c] = v
        rates = []
        for (r, box, (A, B, Dp)), phi in zip(self.faces, aux):
            d = [D[r][c][box] for c in range(9)]
            ev = [e[r][b][box] for b in range(3)]
            lam, mu, slw = self.lam[box], self.mu[box], self.slw[box]
            R = {a: slw * sum(ev[b] * d[STRESS[a][b]] for b in range(3)) for a in range(3)}
            R.update(self._hooke([[ev[b] * d[a] for b in range(3)] for a in range(3)], lam, mu))
            rate = torch.stack([Dp * R[c] - A * phi[c] for c in range(9)])
            for c in range(9):
                h[c][box] += (B - 1) * R[c] - B * phi[c]
            if self.free and r < 2:
                # the surface's dV/dzeta follows this direction's derivatives
                tb = (box[1], box[2])
                mat = self.mats[r][:, :, tb[0], tb[1]]
                dv = [sum(mat[a, b] * d[b][-1] for b in range(3)) for a in range(3)]
                ez = [e[2][b][-1][tb] for b in range(3)]
                t = self._hooke([[ez[b] * dv[a] for b in range(3)] for a in range(3)], lam[-1], mu[-1])
                for c, v in t.items():
                    h[c][nk - 1][tb] += (B[-1] - 1) * v
                    rate[c][-1] += Dp[-1] * v
            rates.append(rate)
        return torch.stack(h), rates

    def shot(self, shot, steps, dt):
        dev, case = self.met.device, self.c
        nz, ny, nx = self.met.shape[1:]
        w = (torch.zeros((9, nz, ny, nx), dtype=torch.float64, device=dev) if shot["w"] is None
             else torch.from_numpy(np.asarray(shot["w"], np.float64)).to(dev))
        aux = [torch.zeros((9,) + tuple(s.stop - s.start for s in box), dtype=torch.float64, device=dev)
               for _, box, _ in self.faces]
        src = shot["src"]
        pt = torch.from_numpy(np.asarray(src["ext_indx"])).to(dev)
        co = torch.from_numpy(np.asarray(src["ext_coef"], np.float64)).to(dev)
        jac = self.met[0].reshape(-1)[pt]
        slw_pad = torch.zeros((nz, ny, nx), dtype=torch.float64, device=dev)
        slw_pad[self.inner] = self.slw
        slw = slw_pad.reshape(-1)[pt]
        idx = torch.from_numpy(shot["idx"]).to(dev)
        fr = torch.from_numpy(np.asarray(shot["frac"], np.float64)).to(dev)
        # corner 5 also takes corner 4's weight, as the recorder defines it
        x, y, z = fr[:, 0], fr[:, 1], fr[:, 2]
        wt = [(1 - x) * (1 - y) * (1 - z), x * (1 - y) * (1 - z), (1 - x) * y * (1 - z), x * y * (1 - z),
              0 * x, (1 - x) * (1 - y) * z + x * (1 - y) * z, (1 - x) * y * z, x * y * z]
        wt = torch.stack(wt, 1)
        seis = torch.zeros((len(idx), 9, steps), dtype=torch.float64, device=dev)
        top = NG + case["nk"] - 1
        pg = torch.zeros((15, ny, nx), dtype=torch.float64, device=dev)
        disp = torch.zeros((3, ny, nx), dtype=torch.float64, device=dev)
        for it in range(steps):
            seis[:, :, it] = torch.stack([(w[c].reshape(-1)[idx] * wt).sum(1) for c in range(9)], 1)
            s, sa = w, aux
            new, newa = w.clone(), [v.clone() for v in aux]
            for st in range(4):
                k, ka = self.rhs(s, sa, tuple((v + st) % 2 for v in PAIRS[it % 8]))
                k = torch.nn.functional.pad(k, (NG,) * 6)
                for c in range(9):
                    flat = k[c].view(-1)
                    if c < 3 and src["F"] is not None:
                        flat.index_add_(0, pt, float(src["F"][c, 0, it, st]) * co * slw / jac)
                    if c >= 3 and src["M"] is not None:
                        flat.index_add_(0, pt, -float(src["M"][c - 3, 0, it, st]) * co / jac)
                b = dt * (1 / 6, 1 / 3, 1 / 3, 1 / 6)[st]
                new += b * k
                newa = [v + b * q for v, q in zip(newa, ka)]
                if st < 3:
                    a = dt * (0.5, 0.5, 1.0)[st]
                    s, sa = w + a * k, [v + a * q for v, q in zip(aux, ka)]
            if case["peak"] and self.free:
                v1, v0 = new[:3, top], w[:3, top]
                acc = ((v1 - v0) / dt).abs()
                disp += 0.5 * (v1 + v0) * dt
                now = []
                for q in (v1, acc, disp):
                    now += [q.square().sum(0).sqrt(), q[:2].square().sum(0).sqrt(), *q.abs()]
                pg = torch.maximum(pg, torch.stack(now))
            w, aux = new, newa
        return seis, w, pg


def exact(case, seed):
    if _device() == "cpu" and case["ni"] * case["nj"] * case["nk"] * case["shots"] > 3e5:
        return None
    m = _inputs(case, seed)
    sch = _Scheme(case, m)
    dt = DT if case["storage"] == "f64" else float(np.float32(DT))
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    out, seis = {}, []
    for n, shot in enumerate(m["shots"]):
        q, w, pg = sch.shot(shot, case["steps"], dt)
        seis.append(q.cpu().numpy())
        if n in _snapshot_shots(case):
            w = w[:, NG:NG + nk, NG:NG + nj, NG:NG + ni]
            j, k = shot["planes"]
            out["plane%d" % n] = w[:, k:k + 1].cpu().numpy()
            out["section%d" % n] = w[:, :, j:j + 1].cpu().numpy()
        if n == 0 and case["peak"] and case["top"] == "free":
            out["peak"] = pg.cpu().numpy()
    out["seismograms"] = np.stack(seis)
    return out
