"""The workloads the framework's speed is measured on.

Each case is one call sequence of a user's program through the ctypes binding
(gpu-wm-next_amd/gwm_amd): whole moist and dry steps, the operators a program
of the host mirror calls one by one, an ensemble, the warm-rain surrogate
(inference and training) and the diagnostics of an output time.  Cases are
dicts of plain values with a "kind" (a function below) and the sizes, type and
options of the call.

A pass that changes its state starts from a copy of the start state
(State.copy_from), as a member restarted from an analysis does, so that every
pass does the same work; the terrain perturbation run and the tracer run go on
from where the last pass left them, as a forecast does.

Inputs are made from the seed with torch and uploaded; exact() computes the
same outputs from them in float64 torch, with the operators written out here.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "gpu-wm-next_amd"))
import gwm_amd as G  # noqa: E402

RD, P0, KAPPA, RV, LV, GRAV = 287.05, 1.0e5, 0.2854, 461.5, 2.5e6, 9.81
CP, EPS = RD / KAPPA, RD / RV
GAMMA = 1.0 / (1.0 - KAPPA)
TRACERS = (16, 17, 18)


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------
def listed():
    return [
        # the warm-rain convection benchmark at its size: two moist steps of
        # the FP32 perturbation form, six acoustic substeps
        dict(name="moist_pert_512", kind="moist", nx=512, ny=512, nz=64, prec=32, pert=True,
             ns=6, dt=0.25, steps=2, graph=False),
        # the same in FP64, a quarter of the domain (the precision reference)
        dict(name="moist_f64_256", kind="moist", nx=256, ny=256, nz=64, prec=64, pert=False,
             ns=6, dt=0.25, steps=2, graph=False),
        # a small case of the regression size, replayed from the step graph:
        # bound by launches and latency
        dict(name="moist_small_graph", kind="moist", nx=64, ny=64, nz=40, prec=32, pert=False,
             ns=3, dt=0.5, steps=4, graph=True),
        # the mountain wave: FP32 perturbation form on terrain, open x sides
        # with a relaxation zone
        dict(name="mountain_pert", kind="mountain", nx=192, ny=192, nz=60, prec=32, pert=True,
             ns=6, dt=0.25, steps=1, open_x=True, open_y=False, boundary="relax"),
        # a ragged mountain domain in FP64 with boundary strips on every side
        # (a regional run driven by an analysis)
        dict(name="mountain_f64", kind="mountain", nx=151, ny=97, nz=40, prec=64, pert=False,
             ns=4, dt=0.5, steps=1, open_x=True, open_y=True, boundary="strips"),
        # the acoustic subcycle alone, flat with open sides, odd sizes
        dict(name="fast_open", kind="fast", nx=331, ny=203, nz=50, prec=32, pert=False, ns=4,
             dt=0.5, open_x=True, open_y=True),
        # the slow tendencies alone
        dict(name="slow_full", kind="slow", nx=500, ny=380, nz=60, prec=32, pert=False,
             open_x=False, open_y=False),
        # tracer transport alone with the winds held
        dict(name="tracers_pert", kind="tracers", nx=300, ny=260, nz=48, prec=32, pert=True,
             dt=2.0),
        # warm rain by the surrogate network in a cloudy domain
        dict(name="surrogate_rain", kind="surrain", nx=256, ny=256, nz=64, pert=False, dt=5.0),
        # one epoch of surrogate training from fixed weights
        dict(name="surrogate_train", kind="train", rows=65536, batch=4096),
        # an ensemble of uneven members advanced together
        dict(name="ensemble", kind="ensemble", members=8, nmin=96, nmax=224, prec=32, ns=4,
             dt=0.5, steps=4, shape_seed=3),
        # the budget sums of an output time
        dict(name="summary", kind="summary", nx=512, ny=512, nz=64, prec=32, pert=False),
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi], odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["moist", "moist", "mountain", "mountain", "fast", "slow", "tracers",
                       "surrain", "train", "ensemble", "summary"])
    nx, ny, nz = _size(rng, 40, 420), _size(rng, 40, 420), rng.randint(24, 64)
    prec = rng.choice([32, 32, 64])
    pert = prec == 32 and rng.random() < 0.5
    if prec == 64 or kind == "mountain":
        nx, ny = min(nx, 224), min(ny, 224)
    dom = dict(nx=nx, ny=ny, nz=nz)
    if kind == "moist":
        graph = rng.random() < 0.4
        return dict(kind=kind, **dom, prec=prec, pert=pert, ns=rng.choice([3, 4, 6]), dt=0.25,
                    steps=4 if graph else 2, graph=graph)
    if kind == "mountain":
        return dict(kind=kind, **dom, prec=prec, pert=pert, ns=rng.choice([3, 4, 6]), dt=0.25,
                    steps=1, open_x=True, open_y=rng.random() < 0.5,
                    boundary=rng.choice(["relax", "strips"]))
    if kind == "fast":
        op = not pert and rng.random() < 0.5
        return dict(kind=kind, **dom, prec=prec, pert=pert, ns=rng.choice([3, 4, 6]), dt=0.25,
                    open_x=op, open_y=op)
    if kind == "slow":
        op = not pert and rng.random() < 0.5
        return dict(kind=kind, **dom, prec=prec, pert=pert, open_x=op, open_y=op)
    if kind == "tracers":
        return dict(kind=kind, **dom, prec=prec, pert=pert, dt=2.0)
    if kind == "surrain":
        return dict(kind=kind, nx=min(nx, 300), ny=min(ny, 300), nz=nz, pert=rng.random() < 0.5,
                    dt=5.0)
    if kind == "train":
        batch = rng.choice([1024, 2048, 4096, 8192])
        return dict(kind=kind, rows=batch * rng.randint(4, 24) + rng.randint(0, 63), batch=batch)
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(3, 8), nmin=64, nmax=192, prec=32,
                    ns=rng.choice([3, 4]), dt=0.25, steps=4, shape_seed=rng.randint(0, 999))
    return dict(kind=kind, **dom, prec=prec, pert=pert)


# --------------------------------------------------------------------------
# Inputs, made in float64 from the seed and rounded to the working precision
# --------------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _levels(nz, terrain):
    """Interfaces: 100 m to 500 m up to 16 km, or 50 m to 600 m up to 20 km
    over terrain (a geometric stretching rescaled to the top)."""
    lo, hi, top = (50.0, 600.0, 20000.0) if terrain else (100.0, 500.0, 16000.0)
    s = np.arange(nz) / max(nz - 1, 1)
    dz = lo * (hi / lo) ** s
    return np.concatenate([[0.0], np.cumsum(dz) * (top / dz.sum())])


def _taper(eta, taper=0.25):
    s = np.clip((eta - taper) / (1.0 - taper), 0.0, 1.0)
    return np.where(eta <= taper, 1.0, np.where(eta >= 1.0, 0.0, 1.0 - s * s * (3.0 - 2.0 * s)))


def _terrain(nx, ny, seed):
    """A ridge along y with a bump on it, 200 m to 500 m high (float32)."""
    r = np.random.RandomState(seed)
    h, a = 200.0 + 300.0 * r.rand(), 8.0 + 6.0 * r.rand()
    x = (np.arange(nx) - 0.5 * nx)[None, :]
    y = (np.arange(ny) - 0.5 * ny)[:, None]
    t = h / (1.0 + (x / a) ** 2) * (1.0 + 0.2 * np.cos(2.0 * np.pi * y / ny))
    return np.ascontiguousarray(t.astype(np.float32))


class _Domain:
    """Grid numbers of a case, as plain float64 arrays."""

    def __init__(self, nx, ny, nz, open_x, open_y, terrain):
        self.nx, self.ny, self.nz, self.open_x, self.open_y = nx, ny, nz, open_x, open_y
        self.dx = self.dy = 1000.0
        self.terrain = terrain
        self.zi = _levels(nz, terrain is not None)
        d = _dev()
        zc = 0.5 * (self.zi[1:] + self.zi[:-1])
        t = torch.zeros((1, 1), dtype=torch.float64, device=d)
        if terrain is not None:
            t = torch.from_numpy(terrain).to(d).double()
        top = self.zi[-1]

        def lift(z):
            col = torch.from_numpy(z).to(d)[:, None, None]
            return col + torch.from_numpy(_taper(z / top)).to(d)[:, None, None] * t[None]

        zf = lift(self.zi)
        self.zc = lift(zc)  # (nz, ny, nx), or (nz, 1, 1) when flat
        self.idz_c = 1.0 / (zf[1:] - zf[:-1])
        self.idz_f = 1.0 / (self.zc[1:] - self.zc[:-1])  # interior faces


def _fields(dom, seed, prec, moist, calm=False):
    """The fields of a developed state over a sounding: rho, rho*theta, the
    face momenta (wind of some m/s with smooth structure and a little noise)
    and, with `moist`, the tracer masses (vapour scaled by U(0.85, 1.25),
    cloud and rain in 30 % of the cells each); `calm`: without the noise.
    Owned values, in the working precision."""
    d = _dev()
    gen = torch.Generator(device=d)
    gen.manual_seed(1000003 * (seed % 100003) + 17)
    nx, ny, nz = dom.nx, dom.ny, dom.nz
    shape = (nz, ny, nx)

    def rand(*s):
        return torch.rand(s, generator=gen, dtype=torch.float64, device=d)

    z = dom.zc.expand(shape)
    if dom.terrain is not None:  # constant N: the Exner function in closed form
        n2, ths = 1.0e-4 * (0.9 + 0.2 * float(rand(1))), 288.0
        th = ths * torch.exp(n2 * z / GRAV)
        ex = 1.0 - GRAV * GRAV / (CP * ths * n2) * (1.0 - torch.exp(-n2 * z / GRAV))
    else:
        zz = np.linspace(0.0, dom.zi[-1], 4001)
        prof = np.where(zz < 12000.0, 300.0 + 43.0 * (zz / 12000.0) ** 1.25, 343.0 *
                        np.exp(GRAV / (CP * 215.0) * (np.maximum(zz, 12000.0) - 12000.0)))
        inv = 1.0 / prof
        exner = 1.0 - GRAV / CP * np.concatenate(
            [[0.0], np.cumsum(0.5 * (inv[1:] + inv[:-1]) * np.diff(zz))])
        zc = dom.zc.cpu().numpy().ravel()
        lev = [torch.from_numpy(np.interp(zc, zz, v)).to(d)[:, None, None].expand(shape)
               for v in (prof, exner)]
        th, ex = lev[0].clone(), lev[1]
        th += (rand(*shape) - 0.5) * torch.exp(-((z / 1500.0) ** 2))
    p = P0 * ex ** (1.0 / KAPPA)
    rho = p / (RD * th * ex)
    noise = 0.0 if calm else 0.2
    x = torch.arange(nx + 1, device=d, dtype=torch.float64) * (2.0 * math.pi / nx)
    y = torch.arange(ny + 1, device=d, dtype=torch.float64) * (2.0 * math.pi / ny)
    amp, ph = 2.0 + 3.0 * rand(4), 2.0 * math.pi * rand(4)
    zu = (dom.zi[-1] - z.mean(dim=(1, 2)))[:, None, None] / dom.zi[-1]
    u = 10.0 + amp[0] * zu * torch.sin(y[None, :ny, None] + ph[0]) * torch.cos(x[None, None] + ph[1])
    v = amp[1] * zu * torch.sin(x[None, None, :nx] + ph[2]) * torch.cos(y[None, :, None] + ph[3])
    u = u * rho.mean(dim=(1, 2))[:, None, None] + noise * (rand(nz, ny, nx + 1) - 0.5)
    v = v * rho.mean(dim=(1, 2))[:, None, None] + noise * (rand(nz, ny + 1, nx) - 0.5)
    w = (noise + 0.01) * (rand(nz + 1, ny, nx) - 0.5)
    w[0] = 0.0
    w[-1] = 0.0
    if not dom.open_x:
        u[..., -1] = u[..., 0]
    if not dom.open_y:
        v[:, -1] = v[:, 0]
    f = {0: rho, 1: rho * th, 2: u, 3: v, 4: w}
    if moist:
        T = th * ex
        rh = torch.clamp(1.0 - 0.75 * (z / 12000.0) ** 1.25, min=0.05)
        qv = torch.clamp(rh * _qsat(T, p), max=0.014)
        qv = qv * (0.85 + 0.4 * rand(*shape))
        qc, qr = (torch.randn(shape, generator=gen, dtype=torch.float64, device=d).abs() * a *
                  (rand(*shape) < 0.3) for a in (1.5e-3, 0.8e-3))
        f.update({16: rho * qv, 17: rho * qc, 18: rho * qr})
    dt = torch.float64 if prec == 64 else torch.float32
    return {k: a.to(dt) for k, a in f.items()}


_CTX = {}


def _ctx(prec):
    """The program's context of a precision (it keeps the tuned shapes)."""
    if prec not in _CTX:
        _CTX[prec] = G.Context(0, G.F64 if prec == 64 else G.F32)
    return _CTX[prec]


def _upload(st, fields):
    for k, a in fields.items():
        s = torch.zeros(st.storage_shape(k), dtype=a.dtype)
        s[:, 1:-1, 1:-1] = a.cpu()
        st.set_storage(k, s.numpy())


class _Fields(dict):
    """Fields of a device state by name.  They stay the state's own buffers
    and come to the host when one is read (FP64 for a perturbation state:
    its departure plus the base)."""

    def __init__(self, st, ids):
        super().__init__({"f%02d" % k: k for k in ids})
        self.st = st

    def __getitem__(self, name):
        k = dict.__getitem__(self, name)
        return self.st.get_f64(k) if self.st.perturbation and k < 2 else self.st.get(k)


def _terrain_of(c, seed):
    return _terrain(c["nx"], c["ny"], seed) if c["kind"] == "mountain" else None


def _domain(c, seed):
    return _Domain(c["nx"], c["ny"], c["nz"], c.get("open_x", False), c.get("open_y", False),
                   _terrain_of(c, seed))


def _grid(dom, prec):
    return G.Grid(_ctx(prec), dom.nx, dom.ny, dom.nz, periodic_x=not dom.open_x,
                  periodic_y=not dom.open_y, dx=dom.dx, dy=dom.dy, z_interfaces=dom.zi,
                  terrain=dom.terrain)


def _inputs(c, seed):
    dom = _domain(c, seed)
    kind = c["kind"]
    moist = kind in ("moist", "tracers", "surrain", "summary", "member")
    return dom, _fields(dom, seed, c.get("prec", 32), moist, calm=kind == "mountain")


def _members(c):
    """Member cases of an ensemble: sizes in steps of 16, 40 to 60 levels."""
    r = np.random.RandomState(c["shape_seed"])
    out = []
    for _ in range(c["members"]):
        nx, ny = (16 * int(v) for v in r.randint(c["nmin"] // 16, c["nmax"] // 16 + 1, 2))
        out.append(dict(kind="member", nx=nx, ny=ny, nz=int(r.choice([40, 48, 60])),
                        prec=c["prec"], pert=False))
    return out


def _weights(seed):
    """FP32 network parameters (Xavier uniform, small biases)."""
    r = np.random.RandomState(seed % 1000003)
    out = []
    for fi, fo in ((7, 64), (64, 64), (64, 64), (64, 4)):
        lim = math.sqrt(6.0 / (fi + fo))
        out += [r.uniform(-lim, lim, fi * fo), 0.1 * r.uniform(-1.0, 1.0, fo)]
    return np.concatenate(out).astype(np.float32)


def _norm(x):
    """Normalisation and fallback box of feature rows x (float64 numpy): the
    1st to 99th percentile, a little wider, so that a feature which is the
    same over a level (the pressure) does not lie on the edge itself."""
    sd = x.std(axis=0)
    sd[sd == 0] = 1.0
    return dict(x_mean=x.mean(axis=0), x_std=sd, y_mean=[0.0] * 4,
                y_std=[2e-4, 2e-4, 5e-5, 0.4], box_lo=np.percentile(x, 1, axis=0) - 1e-3 * sd,
                box_hi=np.percentile(x, 99, axis=0) + 1e-3 * sd)


def _features(f, dt):
    """(T, p, rho, qv, qc, qr, dt) of the fields, float64, (cells, 7)."""
    rho, rt = f[0].double(), f[1].double()
    r = torch.clamp(rho, min=1e-6)
    p = _pressure(rho, rt)
    T = rt / r * (p / P0) ** KAPPA
    q = [torch.clamp(f[t].double() / r, min=0.0) for t in TRACERS]
    return torch.stack([T, p, r] + q + [torch.full_like(T, dt)], -1).reshape(-1, 7)


def _sur_norm(f, dt):
    x = _features(f, dt)
    step = max(1, x.shape[0] // 50000)
    return _norm(x[::step].cpu().numpy())


def _train_rows(c, seed):
    """Feature rows of a cloudy sounding and a smooth four-output target."""
    dom = _Domain(32, 32, 48, False, False, None)
    x = _features(_fields(dom, seed, 32, True), 5.0).cpu().numpy()
    r = np.random.RandomState(seed % 1000003)
    x = x[r.randint(0, x.shape[0], c["rows"])].astype(np.float32)
    n = _norm(x.astype(np.float64))
    t = (x.astype(np.float64) - n["x_mean"]) / n["x_std"]
    m = r.standard_normal((7, 4)) / math.sqrt(7.0)
    y = (np.tanh(t @ m) * np.asarray(n["y_std"])).astype(np.float32)
    return x, y, n


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "train":
        ctx = _ctx(32)
        x, y, norm = _train_rows(c, seed)
        X, Y = G.DeviceArray(ctx, x.shape), G.DeviceArray(ctx, y.shape)
        X.upload(x)
        Y.upload(y)
        sur = G.Surrogate(ctx, 0)
        sur.set_norm(**norm)
        return dict(case=c, sur=sur, x=X, y=Y, w=_weights(seed))
    if kind == "ensemble":
        start, work, grids = [], [], []
        for m, mc in enumerate(_members(c)):
            dom, f = _inputs(mc, seed + m)
            grids.append(_grid(dom, c["prec"]))
            start.append(G.State(grids[-1], 3))
            _upload(start[-1], f)
            work.append(G.State(grids[-1], 3))
        return dict(case=c, start=start, work=work, cfg=G.step_config(c["dt"], c["ns"]),
                    wr=G.warm_rain_config(c["dt"], rain_terminal_velocity=12.0))
    dom, f = _inputs(c, seed)
    grid = _grid(dom, c.get("prec", 32))
    ntr = 3 if 16 in f else 0
    start = G.State(grid, ntr, perturbation=c["pert"])
    _upload(start, f)
    st = dict(case=c, grid=grid, start=start,
              cfg=G.step_config(c.get("dt", 1.0), c.get("ns", 1)),
              wr=G.warm_rain_config(c.get("dt", 1.0), rain_terminal_velocity=12.0))
    if kind in ("moist", "fast", "surrain") or (kind == "mountain" and not c["pert"]):
        st["work"] = G.State(grid, ntr, perturbation=c["pert"])
        st["work"].copy_from(start)
    else:
        st["work"] = start
    if kind == "mountain":
        st["work"].capture_boundary()
        mode, width = (G.BOUNDARY_RELAX, 5.0) if c["boundary"] == "relax" else (G.BOUNDARY_STRIPS, 0.0)
        st["bnd"] = G.BoundaryConfig(mode, width, G.BOUNDARY_FN(), None)
    if kind == "surrain":
        st["sur"] = G.Surrogate(_ctx(32), 0)
        st["sur"].set_norm(**_sur_norm(f, c["dt"]))
        st["sur"].set_params(_weights(seed))
    return st


def run(state):
    s, c = state, state["case"]
    kind, work, start = c["kind"], s.get("work"), s.get("start")
    if kind == "moist":
        work.copy_from(start)
        if c["graph"]:
            work.moist_steps_graph(s["cfg"], s["wr"], c["steps"])
        else:
            for _ in range(c["steps"]):
                work.moist_step(s["cfg"], s["wr"])
        return _Fields(work, (0, 1, 2, 3, 4, 11) + TRACERS)
    if kind == "mountain":
        if work is not start:
            work.copy_from(start)
        for _ in range(c["steps"]):
            work.ssprk3_step(s["cfg"], s["bnd"])
        return _Fields(work, range(5))
    if kind == "fast":
        work.copy_from(start)
        work.fast_modes(s["cfg"])
        return _Fields(work, range(5))
    if kind == "slow":
        work.slow_tendencies(s["cfg"])
        return _Fields(work, range(6, 11))
    if kind == "tracers":
        work.tracers_ssprk3(s["cfg"])
        return _Fields(work, TRACERS)
    if kind == "surrain":
        work.copy_from(start)
        n = work.warm_rain_surrogate(s["wr"], s["sur"])
        return [_Fields(work, (1, 11) + TRACERS), float(n)]
    if kind == "train":
        s["sur"].set_params(s["w"])
        loss = s["sur"].train(s["x"], s["y"], c["rows"], batch=c["batch"], epochs=1)
        return [s["sur"].params(), loss]
    if kind == "ensemble":
        for w, a in zip(work, start):
            w.copy_from(a)
        G.ensemble_steps(work, s["cfg"], s["wr"], c["steps"])
        return [_Fields(w, (0, 1, 2, 3, 4, 11) + TRACERS) for w in work[:6]]
    return _summary_out(work.summary())


_SUMS = ("total_dry_mass", "total_rho_theta_m", "total_horizontal_momentum_x",
         "total_horizontal_momentum_y", "total_vertical_momentum")
_PATHS = ("vapor_path", "cloud_path", "rain_path")
_ENDS = ("rho_min", "rho_max", "theta_min", "theta_max", "u_min", "u_max", "v_min", "v_max",
         "w_min", "w_max")
_QENDS = ("qv_min", "qv_max", "qc_min", "qc_max", "qr_min", "qr_max")


def _summary_out(d):
    out = {n: np.array([d[k] for k in keys]) for n, keys in
           (("sums", _SUMS), ("paths", _PATHS), ("ends", _ENDS), ("mixing", _QENDS))}
    out["nonfinite"] = int(d["nonfinite_values"])
    return out


# --------------------------------------------------------------------------
# Work and tolerances
# --------------------------------------------------------------------------
def _step_elements(ns, moist):
    """Field values a step has to move per cell: each slow stage reads the
    state (and the start state in stages 2 and 3) and writes it; a subcycle's
    first, middle and last substep read and write 6, 9 and 13 fields (faces as
    departures), and its level means take one more pass of two; a tracer stage
    reads rho, three momenta and the tracers and writes them; warm rain reads
    5 and writes 4."""
    sub = 13 if ns == 1 else 6 + 9 * (ns - 2) + 13
    n = (10 + 15 + 15) + 3 * (sub + 2)
    return n + ((4 + 6) + 2 * (4 + 9) + 9 if moist else 0)


def work(case):
    c, kind = case, case["kind"]
    if kind == "train":
        n = (c["rows"] // c["batch"]) * c["batch"]
        mac = 7 * 64 + 2 * 64 * 64 + 64 * 4
        return {"bytes": 44.0 * n, "flops": 6.0 * mac * n}
    if kind == "ensemble":
        cells = sum(m["nx"] * m["ny"] * m["nz"] for m in _members(c))
        n = c["steps"] * _step_elements(c["ns"], True) + 16
        return {"bytes": 4.0 * cells * n, "flops": 8.0 * cells * n}
    cells = c["nx"] * c["ny"] * c["nz"]
    es = 8.0 if c.get("prec", 32) == 64 else 4.0
    if kind in ("moist", "mountain"):
        n = c["steps"] * _step_elements(c["ns"], kind == "moist")
        if kind == "moist":
            n += 16
        elif not c["pert"]:
            n += 10
    elif kind == "fast":
        n = 10 + 3 + 2 + (13 if c["ns"] == 1 else 6 + 9 * (c["ns"] - 2) + 13)
    elif kind == "slow":
        n = 12
    elif kind == "tracers":
        n = 10 + 2 * 13
    elif kind == "surrain":
        return {"bytes": es * cells * (16 + 9), "flops": 18000.0 * cells}
    else:
        n = 8
    return {"bytes": es * cells * n, "flops": 8.0 * cells * n}


def tolerance(case):
    """About four times the error against exact() (which the rounding of the
    working precision sets: in the full FP32 form that of the pressure, whose
    differences are small, dominates the momenta), and 100 times that for the
    largest difference.  A cell of the surrogate case may change sides of the
    training box by rounding."""
    c, kind = case, case["kind"]
    if kind == "train":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "surrain":
        return {"rel": 3e-4, "max": 0.3}
    if kind == "summary":
        return {"rel": 1e-7, "max": 1e-6}
    if c["prec"] == 64:
        rel = 5e-11
    elif kind == "tracers":
        rel = 3e-7
    elif kind == "mountain":
        rel = 3e-5 if c["pert"] else 2e-2
    elif kind == "slow":
        rel = 2e-4 if c["pert"] else 3e-2
    elif kind == "fast":
        rel = 1e-4 if c["pert"] else 1e-3
    else:
        rel = 2e-4
    return {"rel": rel, "max": min(100.0 * rel, 0.9)}


# --------------------------------------------------------------------------
# The same in float64 torch
# --------------------------------------------------------------------------
def _pressure(rho, rt):
    th = rt / torch.clamp(rho, min=1e-6)
    return P0 * torch.clamp(rho * RD * th / P0, min=1e-6) ** GAMMA


def _rho_of(p, th):
    ex = torch.clamp(p / P0, min=1e-6) ** KAPPA
    return p / torch.clamp(RD * th * ex, min=1e-6)


def _qsat(T, p):
    tc = T - 273.15
    es = 611.2 * torch.exp(17.67 * tc / torch.clamp(tc + 243.5, min=1e-6))
    return torch.clamp(EPS * es / torch.clamp(p - (1.0 - EPS) * es, min=1000.0), 0.0, 0.05)


def _up(a, l, r):
    return torch.where(a >= 0, a * l, a * r)


class _Ref:
    """The step's operators on owned arrays (nz, ny, nx) of a domain."""

    def __init__(self, dom):
        self.d = dom

    # neighbour along an axis: wrapped, or `out` beyond an open side
    def nb(self, f, dim, step, out=None):
        g = torch.roll(f, -step, dim)
        if out is not None and (self.d.open_x if dim == -1 else self.d.open_y):
            g = g.clone()
            g.select(dim, -1 if step > 0 else 0).fill_(out)
        return g

    def close(self, f, dim):
        """Full face field from the faces below each cell: the wrap face, or
        closed outer faces."""
        if self.d.open_x if dim == -1 else self.d.open_y:
            f = f.clone()
            f.select(dim, 0).zero_()
            return torch.cat([f, torch.zeros_like(f.narrow(dim, 0, 1))], dim)
        return torch.cat([f, f.narrow(dim, 0, 1)], dim)

    def vgrad(self, p):
        z, g = self.d.zc, torch.empty_like(p)
        g[0] = (p[1] - p[0]) / (z[1] - z[0])
        g[-1] = (p[-1] - p[-2]) / (z[-1] - z[-2])
        g[1:-1] = (p[2:] - p[:-2]) / (z[2:] - z[:-2])
        return g

    def pgf(self, p, dim):
        """Pressure gradient at the lower face of each cell along an axis."""
        h = self.d.dx if dim == -1 else self.d.dy
        g = (p - self.nb(p, dim, -1)) / h
        if self.d.terrain is not None:
            z, v = self.d.zc.expand_as(p), self.vgrad(p)
            g = g - (z - self.nb(z, dim, -1)) / h * 0.5 * (v + self.nb(v, dim, -1))
        return g

    def flux_div(self, q, u, v, w, out):
        """Upwind flux divergence of a cell value q carried by face values."""
        d = self.d
        fx = _up(u[..., :-1], self.nb(q, -1, -1, out), q)
        fx = torch.cat([fx, _up(u[..., -1:], q[..., -1:], self.nb(q, -1, 1, out)[..., -1:])], -1)
        fy = _up(v[:, :-1], self.nb(q, -2, -1, out), q)
        fy = torch.cat([fy, _up(v[:, -1:], q[:, -1:], self.nb(q, -2, 1, out)[:, -1:])], -2)
        lo, hi = torch.cat([q[:1], q]), torch.cat([q, q[-1:]])
        fz = _up(w, lo, hi)
        return ((fx[..., 1:] - fx[..., :-1]) / d.dx + (fy[:, 1:] - fy[:, :-1]) / d.dy +
                (fz[1:] - fz[:-1]) * d.idz_c)

    def slow(self, s):
        d = self.d
        rho, rt, u, v, w = s
        r = torch.clamp(rho, min=1e-6)
        th, p = rt / r, _pressure(rho, rt)
        t_rho = -((u[..., 1:] - u[..., :-1]) / d.dx + (v[:, 1:] - v[:, :-1]) / d.dy +
                  (w[1:] - w[:-1]) * d.idz_c)
        t_rt = -self.flux_div(th, u, v, w, 0.0)
        uc = 0.5 * (u[..., 1:] + u[..., :-1]) / r
        vc = 0.5 * (v[:, 1:] + v[:, :-1]) / r
        wc = 0.5 * (w[1:] + w[:-1]) / r

        def horizontal(q, dim, own, cross, cdim):
            """Tendency of the lower-face momentum along dim."""
            h, hc = (d.dx, d.dy) if dim == -1 else (d.dy, d.dx)
            open_c = d.open_y if dim == -1 else d.open_x
            lo, hi = self.nb(q, dim, -1), self.nb(q, dim, 1)
            if d.open_x if dim == -1 else d.open_y:  # the last face has its own value above
                full = u if dim == -1 else v
                hi = full.narrow(dim, 1, q.shape[dim])
            fw = _up(self.nb(own, dim, -1), lo, q)
            fe = _up(own, q, hi)
            avg = 0.5 * (self.nb(cross, dim, -1) + cross)
            fn = _up(avg, q, self.nb(q, cdim, 1))
            if open_c:
                fn.select(cdim, -1).zero_()
            fs = self.nb(fn, cdim, -1, 0.0)
            aw = 0.5 * (self.nb(wc, dim, -1) + wc)
            ft = torch.zeros_like(q)
            ft[:-1] = _up(aw[:-1], q[:-1], q[1:])
            fb = torch.cat([torch.zeros_like(q[:1]), ft[:-1]])
            idz = d.idz_c.expand_as(q)
            idz = 0.5 * (idz + self.nb(idz, dim, -1))
            a = -((fe - fw) / h + (fn - fs) / hc + (ft - fb) * idz)
            return self.close(a - self.pgf(p, dim), dim)

        t_u = horizontal(u[..., :-1], -1, uc, vc, -2)
        t_v = horizontal(v[:, :-1], -2, vc, uc, -1)
        q = w[1:-1]
        fz = _up(wc, w[:-1], w[1:])
        au, av = 0.5 * (uc[:-1] + uc[1:]), 0.5 * (vc[:-1] + vc[1:])
        fe, fn = _up(au, q, self.nb(q, -1, 1)), _up(av, q, self.nb(q, -2, 1))
        if d.open_x:
            fe[..., -1] = 0.0
        if d.open_y:
            fn[:, -1] = 0.0
        t_w = torch.zeros_like(w)
        a = -((fe - self.nb(fe, -1, -1, 0.0)) / d.dx + (fn - self.nb(fn, -2, -1, 0.0)) / d.dy +
              (fz[1:] - fz[:-1]) * d.idz_f)
        m = th.mean(dim=(1, 2), keepdim=True)
        tf, mf = 0.5 * (th[:-1] + th[1:]), 0.5 * (m[:-1] + m[1:])
        t_w[1:-1] = a + 0.5 * (rho[:-1] + rho[1:]) * (GRAV * (tf - mf) / torch.clamp(mf, min=1e-6))
        return t_rho, t_rt, t_u, t_v, t_w

    def fast(self, rho, th, u, v, w, dt, ns):
        d, dtf = self.d, dt / ns
        du, dv, dw = torch.zeros_like(u), torch.zeros_like(v), torch.zeros_like(w)
        for _ in range(ns):
            p = _pressure(rho, rho * th)
            if d.terrain is None:
                pr = p.mean(dim=(1, 2), keepdim=True)
                rr = rho.mean(dim=(1, 2), keepdim=True)
            else:
                pr, rr = self.column_reference(rho, th, p)
            du = du - dtf * self.close(self.pgf(p, -1), -1)
            dv = dv - dtf * self.close(self.pgf(p, -2), -2)
            pp, rp = p - pr, rho - rr
            dw = dw.clone()
            dw[1:-1] += dtf * (-(pp[1:] - pp[:-1]) * d.idz_f - GRAV * 0.5 * (rp[1:] + rp[:-1]))
            div = ((du[..., 1:] - du[..., :-1]) / d.dx + (dv[:, 1:] - dv[:, :-1]) / d.dy +
                   (dw[1:] - dw[:-1]) * d.idz_c)
            rho = torch.clamp(rho - dtf * div, min=1e-6)
        return rho, rho * th, u + du, v + dv, w + dw

    def column_reference(self, rho, th, p):
        z, thk = self.d.zc, rho * th / torch.clamp(rho, min=1e-6)
        pr, rr = [p[0]], [_rho_of(p[0], thk[0])]
        for k in range(1, p.shape[0]):
            dz = z[k] - z[k - 1]
            pn = torch.clamp(pr[-1] - GRAV * rr[-1] * dz, min=1.0)
            for _ in range(4):
                pn = torch.clamp(pr[-1] - GRAV * 0.5 * (rr[-1] + _rho_of(pn, thk[k])) * dz, min=1.0)
            rr.append(_rho_of(pn, thk[k]))
            pr.append(pn)
        return torch.stack(pr), torch.stack(rr)

    def boundary(self, s, ref, how):
        out = []
        for f, r in zip(s, ref):
            far = torch.full(f.shape[1:], 1e30, dtype=torch.float64, device=f.device)
            for dim, op in ((-1, self.d.open_x), (-2, self.d.open_y)):
                if op:
                    n = f.shape[dim]
                    i = torch.arange(n, device=f.device, dtype=torch.float64)
                    e = torch.minimum(i, n - 1 - i)
                    far = torch.minimum(far, e[None, :] if dim == -1 else e[:, None])
            wgt = (far == 0).double() if how == "strips" else torch.clamp(1.0 - far / 5.0, min=0.0) ** 2
            out.append(f + wgt * (r - f))
        return out

    def step(self, x, dt, ns, how=None, ref=None):
        floor = (1e-6, 1e-6, -1e30, -1e30, -1e30)
        s = self.boundary(x, ref, how) if how else x
        for n, (wa, wb) in enumerate(((0.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0))):
            y = [wa * q + wb * torch.clamp(f + dt * t, min=m)
                 for q, f, t, m in zip(x, s, self.slow(s), floor)]
            th = y[1] / torch.clamp(y[0], min=1e-6)
            s = self.fast(y[0], th, y[2], y[3], y[4], dt, ns)
            if how and n < 2:
                s = self.boundary(s, ref, how)
        return s

    def tracers(self, qs, s, dt):
        r = torch.clamp(s[0], min=1e-6)
        out = []
        for q0 in qs:
            q = q0
            for wa, wb in ((0.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0)):
                q = wa * q0 + wb * torch.clamp(q - dt * self.flux_div(q / r, s[2], s[3], s[4], 0.0),
                                               min=0.0)
            out.append(q)
        return out

    def warm_rain(self, rho, rt, qs, dt, vt, network=None):
        """Source terms (thresholds, relaxation and rates of the default
        configuration), then fallout; network(features) -> (changes, where)
        takes its cells' changes instead.  Returns rt, tracers, bucket."""
        r = torch.clamp(rho, min=1e-6)
        th, p = rt / r, _pressure(r, rt)
        T = th * (p / P0) ** KAPPA
        lf = LV / (CP * torch.clamp(T / th, min=1e-6))
        qv, qc, qr = (torch.clamp(q / r, min=0.0) for q in qs)
        v0, c0, r0, th0 = qv, qc, qr, th
        qs1 = _qsat(T, p)
        cnd = torch.where(qv > qs1, torch.minimum(qv - qs1, qv), -torch.minimum(qs1 - qv, qc))
        qv, qc, th = qv - cnd, qc + cnd, th + lf * cnd
        exc = torch.clamp(qc - 1e-4, min=0.0)
        cv = torch.minimum(exc, dt * 1e-3 * exc)
        qc, qr = qc - cv, qr + cv
        p2 = _pressure(r, r * th)
        qs2 = _qsat(th * (p2 / P0) ** KAPPA, p2)
        e = torch.where(qv < qs2, torch.minimum(qr, dt * 5e-3 * torch.minimum(qs2 - qv, qr)), 0.0)
        qr, qv, th = qr - e, qv + e, th - lf * e
        qv, qc, qr = (torch.clamp(q, min=0.0) for q in (qv, qc, qr))
        outside = 0.0
        if network is not None:
            f = torch.stack([T, p, r, v0, c0, r0, torch.full_like(T, dt)], -1)
            dc, dr, dth, inbox = network(f)
            quiet = (c0 <= 0) & (r0 <= 0) & (v0 <= qs1)
            outside = float((~inbox).sum())
            dc, dr = torch.maximum(dc, -c0), torch.maximum(dr, -r0)
            dv = -(dc + dr)
            lam = torch.where(v0 + dv < 0, v0 / torch.clamp(-dv, min=1e-30), 1.0)
            net = inbox & ~quiet
            qv = torch.where(net, torch.clamp(v0 + lam * dv, min=0.0), torch.where(quiet, v0, qv))
            qc = torch.where(net, torch.clamp(c0 + lam * dc, min=0.0), torch.where(quiet, c0, qc))
            qr = torch.where(net, torch.clamp(r0 + lam * dr, min=0.0), torch.where(quiet, r0, qr))
            th = torch.where(net, th0 + lam * dth, torch.where(quiet, th0, th))
        idz = self.d.idz_c.expand_as(rho)
        rqr, inc = r * qr, torch.zeros_like(rho[0])
        out = []
        for k in range(rho.shape[0] - 1, -1, -1):
            old = torch.clamp(rqr[k], min=0.0) / idz[k]
            fall = torch.clamp(vt * dt * idz[k], 0.0, 1.0) * old
            out.append((old - fall + inc) * idz[k])
            inc = fall
        return r * th, [r * qv, r * qc, torch.stack(out[::-1])], inc[None], outside


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _layers(p):
    out, at = [], 0
    for fi, fo in ((7, 64), (64, 64), (64, 64), (64, 4)):
        out.append((p[at:at + fi * fo].reshape(fi, fo), p[at + fi * fo:at + fi * fo + fo]))
        at += fi * fo + fo
    return out


def _mlp(x, p):
    for n, (w, b) in enumerate(_layers(p)):
        x = x @ w + b
        if n < 3:
            x = _gelu(x)
    return x


def _norm32(n):
    """The normalisation as the network holds it (FP32), in float64."""
    return {k: torch.from_numpy(np.asarray(v, np.float32)).double().to(_dev()) for k, v in n.items()}


def _exact_train(c, seed):
    x, y, norm = _train_rows(c, seed)
    n = _norm32(norm)
    x, y = (torch.from_numpy(a).double().to(_dev()) for a in (x, y))
    x, y = (x - n["x_mean"]) / n["x_std"], (y - n["y_mean"]) / n["y_std"]
    p = torch.from_numpy(_weights(seed)).double().to(_dev()).requires_grad_(True)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    steps, loss = c["rows"] // c["batch"], 0.0
    b1, b2, eps = (float(np.float32(a)) for a in (0.9, 0.999, 1e-8))
    for s in range(steps):
        at = slice(s * c["batch"], (s + 1) * c["batch"])
        lr = 1e-4 + (2e-3 - 1e-4) * 0.5 * (1.0 + math.cos(math.pi * s / steps))
        l = ((_mlp(x[at], p) - y[at]) ** 2).mean()
        g, = torch.autograd.grad(l, p)
        loss += float(l.detach())
        m, v = b1 * m + (1.0 - b1) * g, b2 * v + (1.0 - b2) * g * g
        c1, c2 = 1.0 - b1 ** (s + 1), 1.0 - b2 ** (s + 1)
        p = (p.detach() - lr * (m / c1) / (torch.sqrt(v / c2) + eps)).requires_grad_(True)
    return [p.detach().cpu().numpy(), np.array([loss / steps])]


def _host(ids, arrays):
    return {"f%02d" % k: a.cpu().numpy() for k, a in zip(ids, arrays)}


def _exact_moist(c, seed, dt, ns, steps):
    dom, f = _inputs(c, seed)
    ref = _Ref(dom)
    f = {k: a.double() for k, a in f.items()}
    s, q, rain = [f[k] for k in range(5)], [f[k] for k in TRACERS], 0.0
    for _ in range(steps):
        s = list(ref.step(s, dt, ns))
        q = ref.tracers(q, s, dt)
        s[1], q, inc, _ = ref.warm_rain(s[0], s[1], q, dt, 12.0)
        rain = rain + inc
    return _host((0, 1, 2, 3, 4, 11) + TRACERS, s + [rain] + q)


def exact(case, seed):
    c, kind = case, case["kind"]
    with torch.no_grad():
        if kind == "moist":
            return _exact_moist(c, seed, c["dt"], c["ns"], c["steps"])
        if kind == "ensemble":
            return [_exact_moist(mc, seed + m, c["dt"], c["ns"], c["steps"])
                    for m, mc in enumerate(_members(c)[:6])]
        if kind != "train":
            dom, f = _inputs(c, seed)
            ref = _Ref(dom)
            f = {k: a.double() for k, a in f.items()}
            s = [f[k] for k in range(5)]
    if kind == "train":
        return _exact_train(c, seed)
    with torch.no_grad():
        if kind == "mountain":
            for _ in range(c["steps"]):
                s = ref.step(s, c["dt"], c["ns"], c["boundary"], [f[k] for k in range(5)])
            return _host(range(5), s)
        if kind == "fast":
            th = s[1] / torch.clamp(s[0], min=1e-6)
            return _host(range(5), ref.fast(s[0], th, s[2], s[3], s[4], c["dt"], c["ns"]))
        if kind == "slow":
            return _host(range(6, 11), ref.slow(s))
        if kind == "tracers":
            return _host(TRACERS, ref.tracers([f[k] for k in TRACERS], s, c["dt"]))
        if kind == "surrain":
            n = _norm32(_sur_norm(_inputs(c, seed)[1], c["dt"]))
            p = torch.from_numpy(_weights(seed)).double().to(_dev())

            def network(x):
                inbox = ((x >= n["box_lo"]) & (x <= n["box_hi"])).all(-1)
                y = _mlp((x - n["x_mean"]) / n["x_std"], p) * n["y_std"] + n["y_mean"]
                return y[..., 1], y[..., 2], y[..., 3], inbox

            rt, q, rain, outside = ref.warm_rain(s[0], s[1], [f[k] for k in TRACERS], c["dt"], 12.0,
                                                 network)
            return [_host((1, 11) + TRACERS, [rt, rain] + q), outside]
        return _exact_summary(dom, f)


def _exact_summary(dom, f):
    r = torch.clamp(f[0], min=1e-12)
    ends = [f[0], f[1] / r, f[2], f[3], f[4]]
    q = [f[t] for t in TRACERS]
    pair = lambda v: [float(v.min()), float(v.max())]  # noqa: E731
    return {"sums": np.array([float(f[k].sum()) for k in range(5)]),
            "paths": np.array([float((a / dom.idz_c).sum()) for a in q]),
            "ends": np.array(sum((pair(a) for a in ends), [])),
            "mixing": np.array(sum((pair(a / r) for a in q), [])),
            "nonfinite": 0}
