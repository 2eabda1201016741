"""Performance cases: the calls a seismic modelling or inversion program makes
into this framework, at the sizes of its own configurations (201x301, 301x921
and 501x1501 grids, their coarse 251x751 one) and at odd sizes between.

The number of time steps is shortened against a production run (2000 to 6000):
every step costs the same, so a few hundred show the same rates."""
import math

import numpy as np
import torch

from swfwi_amd import capi
from swfwi_amd.batch import Batch, Group, Net
from swfwi_amd.enkf import Enkf

DT = 0.001
VMIN, VMAX = 1500.0, 4500.0
EXACT, FP32 = capi.PREC_EXACT, capi.PREC_FP32


def listed():
    return [
        # one leapfrog step through the drop-in symbol, fields in host memory:
        # a program that keeps its own time loop (the smallest call)
        {"name": "step_201x301", "kind": "step", "nx": 301, "nz": 201, "nb": 20, "damped": True, "prec": EXACT},
        # one shot on a small grid: survey design, a single trial model
        {"name": "forward_201x301", "kind": "forward", "nx": 301, "nz": 201, "nb": 20, "dx": 10.0, "nt": 800,
         "ns": 11, "shot": 5, "prec": EXACT},
        # an encoded supershot in the pure FP32 mode
        {"name": "forward_301x921_fp32", "kind": "forward", "nx": 921, "nz": 301, "nb": 30, "dx": 12.5, "nt": 800,
         "ns": 60, "shot": -1, "prec": FP32},
        # the adjoint gradient of an encoded supershot, bit-exact mode
        {"name": "gradient_301x921", "kind": "gradient", "nx": 921, "nz": 301, "nb": 30, "dx": 12.5, "nt": 800,
         "ns": 60, "shot": -1, "prec": EXACT},
        # the adjoint gradient of one shot on the largest grid
        {"name": "gradient_501x1501", "kind": "gradient", "nx": 1501, "nz": 501, "nb": 30, "dx": 12.5, "nt": 700,
         "ns": 16, "shot": 7, "prec": EXACT},
        # observed data of a whole survey, every shot at once
        {"name": "shots_301x921", "kind": "shots", "nx": 921, "nz": 301, "nb": 30, "dx": 12.5, "nt": 400, "ns": 60,
         "prec": EXACT},
        # one epoch of encoded-source inversion: gradient, line search, update
        {"name": "ess_301x921", "kind": "ess", "nx": 921, "nz": 301, "nb": 30, "dx": 12.5, "nt": 800, "ns": 24,
         "prec": EXACT},
        # one epoch of shot-by-shot inversion of a small survey
        {"name": "fwi_201x301", "kind": "fwi", "nx": 301, "nz": 201, "nb": 20, "dx": 10.0, "nt": 700, "ns": 11,
         "prec": EXACT},
        # one ensemble Kalman analysis: every member's forward run, the FP64
        # data-space products, the update of the members
        {"name": "enkf_201x301_n60", "kind": "enkf", "nx": 301, "nz": 201, "nb": 20, "dx": 10.0, "nt": 500, "ns": 11,
         "members": 60, "prec": EXACT},
        # gradients of 112 shots of three grid sizes in one batch, FP16
        # checkpoints (forward, adjoint source, backward)
        {"name": "batch_mixed_fp16", "kind": "batch", "nx": 301, "nz": 201, "nb": 20, "dx": 10.0, "nt": 480,
         "models": 4, "ns": 16, "nx2": 921, "nz2": 301, "nb2": 30, "nt2": 560, "models2": 2, "nx3": 1501, "nz3": 501,
         "nb3": 30, "nt3": 640, "models3": 1, "snap": capi.SNAP_F16},
        # the coarse 4th-order propagation of 16 shots with the learned
        # correction every 4 steps, and its gradient
        {"name": "coarse_learned_251x751", "kind": "coarse", "nx": 751, "nz": 251, "nb": 15, "dx": 25.0, "nt": 360,
         "ns": 16, "snap": capi.SNAP_F16},
        # 20 training steps of the correction network from given weights
        {"name": "train_161x80", "kind": "train", "nx": 93, "nz": 52, "samples": 256, "batch": 16, "steps": 20},
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    """One more case: any kind, any grid between a small test model and the
    501x1501 one, no dearer than the dearest listed case of its kind."""
    kind = rng.choice(["step", "forward", "forward", "gradient", "gradient", "shots", "ess", "fwi", "enkf", "batch",
                       "coarse", "train"])
    c = {"kind": kind, "nx": _log(rng, 90, 1501), "nz": _log(rng, 60, 501), "nb": rng.randint(12, 34),
         "dx": rng.choice([10.0, 12.5, 15.0]), "prec": rng.choice([EXACT, EXACT, FP32])}
    pts = lambda: (c["nx"] + 2 * c["nb"]) * (c["nz"] + c["nb"])  # noqa: E731
    fit = lambda limit, most: max(1, min(most, int(limit / pts())))  # noqa: E731
    if kind == "step":
        c.pop("dx")
        c["damped"] = rng.random() < 0.7
    elif kind in ("forward", "gradient"):
        c.update(nt=rng.randint(420, 700), ns=rng.randint(1, 40))
        c["shot"] = rng.choice([-1, rng.randrange(c["ns"])])
    elif kind == "shots":
        c.update(nt=rng.randint(320, 400), ns=rng.randint(1, fit(1.9e7, 48)))
    elif kind == "ess":
        c.update(nx=_log(rng, 90, 900), nz=_log(rng, 60, 300))
        c.update(nt=rng.randint(420, 700), ns=rng.randint(2, 20), prec=EXACT)
    elif kind == "fwi":
        c.update(nx=_log(rng, 90, 301), nz=_log(rng, 60, 201))
        c.update(nt=rng.randint(420, 600), ns=rng.randint(1, fit(8e5, 11)), prec=EXACT)
    elif kind == "enkf":
        c.update(nx=_log(rng, 90, 301), nz=_log(rng, 60, 201))
        c.update(nt=rng.randint(320, 480), ns=rng.randint(2, 11), members=rng.randint(8, 56), prec=EXACT)
    elif kind == "batch":
        c.pop("prec")
        c.update(nt=rng.randint(420, 460), models=rng.randint(1, 3), ns=rng.randint(1, fit(6e6, 14)))
        if rng.random() < 0.6:
            c.update(nx2=_log(rng, 90, 600), nz2=_log(rng, 60, 300), nb2=rng.randint(12, 34),
                     nt2=c["nt"] + rng.randint(1, 90), models2=1)
        c["snap"] = rng.choice([capi.SNAP_F32, capi.SNAP_BF16, capi.SNAP_F16])
    elif kind == "coarse":
        c.pop("prec")
        c.update(nx=_log(rng, 90, 751), nz=_log(rng, 60, 251), nb=rng.randint(10, 16), dx=25.0)
        c.update(nt=rng.randint(240, 340), ns=rng.randint(1, 14), snap=rng.choice([capi.SNAP_F32, capi.SNAP_F16]))
    else:
        c = {"kind": kind, "nx": rng.randint(40, 112), "nz": rng.randint(40, 90), "samples": rng.randint(40, 200),
             "batch": rng.randint(2, 16), "steps": rng.randint(5, 18)}
    return c


# ---- inputs -----------------------------------------------------------------


def _model(nx, nz, seed, smooth=False):
    """Velocity in m/s [nx][nz]: depth gradient, dipping layers, a smooth
    random field; `smooth` leaves the layers out (a starting model)."""
    r = np.random.default_rng(seed)
    x, z = np.arange(nx)[:, None] / nx, np.arange(nz)[None, :] / nz
    v = 1800.0 + 1900.0 * z + 0.0 * x
    for k in range(6):
        z0, dip, dv, a, b, ph = r.uniform(0.1, 0.95), r.uniform(-0.1, 0.1), *r.uniform(-250, 250, 1), *r.uniform(1, 5, 2), \
            r.uniform(0, 6.28)
        v = v + 60.0 * np.sin(a * 3 * x + b * 3 * z + ph)
        if not smooth:
            v = v + dv * (z >= z0 + dip * (x - 0.5))
    return np.clip(v, VMIN, VMAX).astype(np.float32)


def _padded(v, nb, dx, dt):
    """The padded model in transformed units dx^2 / (v^2 dt^2)."""
    p = np.pad(v.astype(np.float64), ((nb + 6, nb + 6), (6, nb + 6)), mode="edge")
    return (dx * dx / (p * p * dt * dt)).astype(np.float32)


def _ricker(nt, fm, dt):
    t = np.arange(nt) * dt - 1.0 / fm
    a = (math.pi * fm * t) ** 2
    return ((1 - 2 * a) * np.exp(-a)).astype(np.float32)


def _fm(dx):
    return 1500.0 / dx / 10.0  # ten cells a wavelength at the slowest velocity


def _traces(nt, ng, n, fm, dt, seed):
    """[n][nt][ng] records: Ricker arrivals along seeded hyperbolas."""
    g = torch.Generator().manual_seed(seed)
    t = torch.arange(nt, device="cuda", dtype=torch.float32)[None, :, None] * dt
    x = torch.linspace(0, 1, ng, device="cuda")[None, None, :]
    out = torch.zeros((n, nt, ng), device="cuda")
    for _ in range(3):
        x0, t0, m, a = (torch.rand((n, 1, 1), generator=g).cuda() for _ in range(4))
        tau = torch.sqrt((0.05 + 0.7 * nt * dt * t0) ** 2 + (0.6 * m * (x - x0)) ** 2)
        w = (math.pi * fm * (t - tau)) ** 2
        out += (0.1 + a) * (1 - 2 * w) * torch.exp(-w)
    return out.cpu().numpy()


def _survey(c):
    ns = c["ns"]
    sx = np.linspace(0, c["nx"] - 1, ns + 2)[1:-1].astype(np.int32)
    return sx, np.ones(ns, np.int32), np.arange(c["nx"], dtype=np.int32), np.zeros(c["nx"], np.int32)


def _solver(c):
    sx, sz, gx, gz = _survey(c)
    return capi.Solver(c["nx"], c["nz"], c["nb"], DT, c["dx"], _fm(c["dx"]), c["nt"], sx, sz, gx, gz, c["prec"])


def _source(c, seed):
    """The amplitude table of a call: one wavelet, or a +-1 encoded one per source."""
    w = _ricker(c["nt"], _fm(c["dx"]), DT)
    if c.get("shot", 0) >= 0:
        return w * np.float32(1 + 0.1 * (seed % 7))
    code = np.random.default_rng(seed).integers(0, 2, c["ns"]) * 2 - 1
    return np.ascontiguousarray(w[:, None] * code[None, :].astype(np.float32))


def _wave(c, seed):
    """Two successive smooth fields of a padded grid, zero on its 6-cell rim."""
    nx, nz = c["nx"] + 2 * c["nb"] + 12, c["nz"] + c["nb"] + 12
    r = np.random.default_rng(seed)
    x, z = np.arange(nx)[:, None], np.arange(nz)[None, :]
    modes = [(*r.uniform(0.05, 0.5, 2), *r.uniform(0, 6, 2)) for _ in range(4)]
    f = []
    for ph in (0.0, 0.12):
        a = sum(np.sin(kx * x + p + ph) * np.sin(kz * z + q) for kx, kz, p, q in modes)
        a[:6] = a[-6:] = 0
        a[:, :6] = a[:, -6:] = 0
        f.append(a.astype(np.float32))
    return f


def _groups(c, dt):
    out = []
    for k in ("", "2", "3"):
        if "nx" + k not in c:
            continue
        sx = np.linspace(0, c["nx" + k] - 1, c["ns"] + 2)[1:-1].astype(np.int32)
        out.append(Group(c["nx" + k], c["nz" + k], c["nb" + k], c["dx"], dt, _fm(c["dx"]), c["nt" + k], sx,
                         np.ones_like(sx), 0, c["nx" + k], 0, c.get("models" + k, 1),
                         2.0 if c["kind"] == "coarse" else 1.0))
    return out


def _batch_models(c, groups, seed):
    return [[_padded(_model(g.nx, g.nz, seed * 10 + m), g.nb, g.dx, g.dt) for m in range(g.nmodels)] for g in groups]


def _batch_data(groups, seed):
    d = [_traces(g.nt, g.ng, g.nmodels * g.ns, g.fm, g.dt, seed * 10 + k).ravel() for k, g in enumerate(groups)]
    return np.concatenate(d)


def _weights(seed):
    r = np.random.default_rng(seed)
    return np.concatenate([r.standard_normal(288) * math.sqrt(2 / 18), r.standard_normal(2304) * math.sqrt(2 / 144),
                           r.standard_normal(144) * 4e-4]).astype(np.float32)


def _training(c, seed):
    """Fields, their models (squared Courant numbers) and the targets."""
    r = np.random.default_rng(seed)
    n, nx, nz = c["samples"], c["nx"], c["nz"]
    x, z = np.arange(nx, dtype=np.float32)[None, :, None], np.arange(nz, dtype=np.float32)[None, None, :]
    u = lambda a, b: r.uniform(a, b, (n, 1, 1)).astype(np.float32)  # noqa: E731
    p = u(0.3, 1) * np.sin(u(0.3, 1.2) * x + u(0, 6)) * np.sin(u(0.3, 1.2) * z + u(0, 6))
    p = p * np.exp(-(((x - u(0.2, 0.8) * nx) / 20) ** 2) - ((z - u(0.2, 0.8) * nz) / 20) ** 2)
    q = (0.05 + 0.15 * z / nz + 0.02 * np.sin(0.1 * x + u(0, 6))).astype(np.float32)
    q = np.ascontiguousarray(np.broadcast_to(q, p.shape))
    t = p + 0.02 * q * (np.roll(p, 1, 1) - 2 * p + np.roll(p, -1, 1))
    return np.ascontiguousarray(p), q, np.ascontiguousarray(t.astype(np.float32))


# ---- what a program holds before the call ------------------------------------


def prepare(case, seed):
    c, k = dict(case), case["kind"]
    s = {"case": c}
    if k == "step":
        prev, cur = _wave(c, seed)
        s.update(prev=prev, cur=cur, vel=_padded(_model(c["nx"], c["nz"], seed), c["nb"], 10.0, DT),
                 u2=np.zeros_like(prev))
    elif k in ("forward", "gradient", "shots"):
        s["solver"] = _solver(c)
        s["solver"].bind_velocity(_padded(_model(c["nx"], c["nz"], seed), c["nb"], c["dx"], DT))
        s["src"] = _source(c, seed)
        if k == "gradient":
            s["vsrc"] = _traces(c["nt"], c["nx"], 1, _fm(c["dx"]), DT, seed)[0]
    elif k in ("ess", "fwi"):
        s["solver"] = _solver(c)
        w = _ricker(c["nt"], _fm(c["dx"]), DT)
        s["solver"].bind_velocity(_padded(_model(c["nx"], c["nz"], seed), c["nb"], c["dx"], DT))
        dobs = s["solver"].forward_shots(w)
        s["start"] = _padded(_model(c["nx"], c["nz"], seed, True), c["nb"], c["dx"], DT)
        s["inv"] = capi.Inversion(s["solver"], w, dobs, VMIN, VMAX, 5, 200.0)
    elif k == "enkf":
        s["solver"] = _solver(c)
        base = _model(c["nx"], c["nz"], seed, True)
        s["solver"].bind_velocity(_padded(_model(c["nx"], c["nz"], seed), c["nb"], c["dx"], DT))
        w = _ricker(c["nt"], _fm(c["dx"]), DT)
        dobs = s["solver"].forward_shots(w)
        s["enkf"] = Enkf(s["solver"], w, dobs, 0.05, c["members"])
        s["members"] = np.stack([_padded(base * np.float32(0.97 + 0.06 * m / c["members"]) + _model(
            c["nx"], c["nz"], seed * 100 + m, True) * np.float32(0.02), c["nb"], c["dx"], DT)
            for m in range(c["members"])])
    elif k in ("batch", "coarse"):
        groups = _groups(c, 2 * DT if k == "coarse" else DT)
        b = Batch(groups, c["snap"], capi.ORDER_4 if k == "coarse" else capi.ORDER_10)
        for gi, ms in enumerate(_batch_models(c, groups, seed)):
            for m, v in enumerate(ms):
                b.bind_model(gi, m, v)
        if k == "coarse":
            s["net"] = Net(_weights(seed))
            b.set_correction(s["net"])
        s.update(batch=b, dobs=_batch_data(groups, seed))
    else:
        p, q, t = _training(c, seed)
        s["net"] = Net(_weights(seed))
        s["net"].set_data(p, q, t, [5, c["nx"] - 5, 5, c["nz"] - 5])
        s["weights"] = _weights(seed)
    return s


# ---- one pass -----------------------------------------------------------------


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "step":  # the program's own leapfrog: step, then swap the levels
        if c["damped"]:
            capi.step_damped(s["prev"], s["cur"], s["vel"], s["u2"], c["nb"] + 6, c["prec"])
        else:
            capi.step_undamped(s["prev"], s["cur"], s["vel"], s["u2"], c["prec"])
        s["prev"], s["cur"] = s["cur"], s["prev"]
        return {"next": s["cur"], "u2": s["u2"]}
    if k == "forward":
        return s["solver"].forward_modeling(s["src"], c["shot"])
    if k == "gradient":
        return s["solver"].calgradient(s["src"], s["vsrc"], c["shot"])
    if k == "shots":
        return s["solver"].forward_shots(s["src"])
    if k in ("ess", "fwi"):  # an inversion's first epoch from its starting model
        s["solver"].bind_velocity(s["start"])
        s["inv"].ess_epoch(0) if k == "ess" else s["inv"].fwi_epoch(0)
        st = s["inv"].stats()
        return {"gradient": s["inv"].gradient(), "model": s["solver"].velocity(), "objective": st["obj1"],
                "step": st["steplen"]}
    if k == "enkf":
        s["enkf"].set_members(s["members"])
        s["enkf"].analyze(None, 7)
        return {"members": s["enkf"].members(), "mean": s["enkf"].mean()}
    if k in ("batch", "coarse"):
        b = s["batch"]
        b.forward(want_data=False)
        vsrc = b.adjoint_source(s["dobs"], want=k == "coarse")
        _, g = b.backward(None, want_entries=False)
        return {"gradient": g, "vsrc": vsrc} if k == "coarse" else {"gradient": g}
    s["net"].set_weights(s["weights"])
    losses = s["net"].train(c["batch"], c["steps"], 1e-3, 3)
    return {"weights": s["net"].weights(), "losses": losses}


# ---- what a pass cannot do without ---------------------------------------------

STEP_FLOPS, COARSE_FLOPS, NET_FLOPS = 45, 25, 5472  # per point: a 10th-order step, a 4th-order one, the network


def work(case):
    c, k = case, case["kind"]
    if k == "train":
        n = (c["nx"] - 10) * (c["nz"] - 10) * c["batch"] * c["steps"]
        return {"bytes": 12.0 * c["nx"] * c["nz"] * c["batch"] * c["steps"], "flops": 3.0 * NET_FLOPS * n}
    upd = lambda q="": float((c["nx" + q] + 2 * c["nb" + q]) * (c["nz" + q] + c["nb" + q]))  # noqa: E731
    fld = lambda q="": 4.0 * (c["nx" + q] + 2 * c["nb" + q] + 12) * (c["nz" + q] + c["nb" + q] + 12)  # noqa: E731
    p, f = upd(), fld()
    if k == "step":
        return {"bytes": 5 * f, "flops": STEP_FLOPS * p}
    if k in ("batch", "coarse"):
        b = fl = 0.0
        for q in ("", "2", "3"):
            if "nx" + q in c:
                n, nt, m = c["ns"] * c.get("models" + q, 1), c["nt" + q], c.get("models" + q, 1)
                last = 304 if k == "batch" else 152
                fl += n * upd(q) * (nt + nt - last) * (STEP_FLOPS if k == "batch" else COARSE_FLOPS)
                if k == "coarse":
                    fl += n * upd(q) * NET_FLOPS * 2 * (nt // 4)
                b += 2 * m * fld(q) + 4.0 * n * nt * c["nx" + q] * (1 if k == "batch" else 2)
        return {"bytes": b, "flops": fl}
    data, back = 4.0 * c["nt"] * c["nx"], c["nt"] - 301
    if k == "forward":
        return {"bytes": f + data, "flops": STEP_FLOPS * p * c["nt"]}
    if k == "gradient":
        return {"bytes": 2 * f + data, "flops": STEP_FLOPS * p * (c["nt"] + 2 * back)}
    if k == "shots":
        return {"bytes": f + data * c["ns"], "flops": STEP_FLOPS * p * c["nt"] * c["ns"]}
    if k == "ess":
        return {"bytes": 3 * f + data * c["ns"], "flops": STEP_FLOPS * p * (3 * c["nt"] + 2 * back)}
    if k == "fwi":
        return {"bytes": 3 * f + data * c["ns"], "flops": STEP_FLOPS * p * c["ns"] * (3 * c["nt"] + 2 * back)}
    n = c["members"]
    return {"bytes": 2 * n * f + data * c["ns"], "flops": STEP_FLOPS * p * c["nt"] * n + 6.0 * n * n * c["nt"] * c["nx"]}


# ---- the same in 64 bits ---------------------------------------------------------

A = [float(np.float32(a)) for a in (1.53400796, 1.78858721, -0.31660756, 0.07612173, -0.01626042, 0.00216736)]


class _Fd:
    """The leapfrog step on [entries][nx][nz] fields in FP64."""

    def __init__(self, vel, nb, order=10, dscale=1.0):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        vel = torch.as_tensor(vel, device=self.dev)
        self.rv = 1.0 / vel.double()
        self.rv = self.rv if self.rv.dim() == 3 else self.rv[None]
        _, nx, nz = self.rv.shape
        d = torch.zeros((nx, nz), dtype=torch.float64, device=self.dev)
        k = torch.arange(nb, dtype=torch.float64, device=self.dev)
        d[:nb] = (0.05 * ((nb - k) / nb) ** 2)[:, None]
        d[nx - nb:] = (0.05 * ((k + 1) / nb) ** 2)[:, None]
        d[:, nz - nb:] = (0.05 * ((k + 1) / nb) ** 2)[None, :]
        d = (d * dscale)[6:-6, 6:-6]
        self.a, self.b, self.order = 2 - 2 * d + d * d, 1 - 2 * d, order
        self.r = self.rv[:, 6:-6, 6:-6]

    def lap(self, p):  # on [5, n-5)
        n, m = p.shape[1], p.shape[2]
        at = lambda i, j: p[:, 5 + i:n - 5 + i, 5 + j:m - 5 + j]  # noqa: E731
        if self.order == 10:
            u = -4.0 * A[0] * at(0, 0)
            w = A
        else:
            u = -5.0 * at(0, 0)
            w = [0, 4.0 / 3, -1.0 / 12]
        for k in range(1, len(w)):
            u += w[k] * (at(0, -k) + at(0, k) + at(-k, 0) + at(k, 0))
        return u

    def step(self, cur, prev, damped=True):
        """prev <- next"""
        u = self.lap(cur)
        c, p, u0 = cur[:, 6:-6, 6:-6], prev[:, 6:-6, 6:-6], u[:, 1:-1, 1:-1]
        n = (self.a * c - self.b * p if damped else 2 * c - p) + self.r * u0
        if self.order == 10:
            n += self.r * self.r / 12 * (u[:, 1:-1, :-2] + u[:, 1:-1, 2:] + u[:, :-2, 1:-1] + u[:, 2:, 1:-1] - 4 * u0)
        prev[:, 6:-6, 6:-6] = n
        return u

    def zeros(self, n):
        return torch.zeros((n,) + self.rv.shape[1:], dtype=torch.float64, device=self.dev)


def _taper(nt, dt):
    w = np.zeros(nt)
    for it in range(nt - 1, -1, -1):
        t = float(np.float32(dt)) * it
        if t > 0.4:
            w[it] = 1
        elif t > 0.3:
            w[it] = (t - 0.3) / 0.1
        else:
            break
    return w


def _exact_shots(c, seed, gradient=False):
    """Seismograms [entries][nt][ng], or the gradient, of a solver case."""
    fd = _Fd(_padded(_model(c["nx"], c["nz"], seed), c["nb"], c["dx"], DT), c["nb"] + 6)
    sx, sz, gx, gz = (torch.as_tensor(a.astype(np.int64), device=fd.dev) for a in _survey(c))
    sx, sz, gx, gz = sx + c["nb"] + 6, sz + 6, gx + c["nb"] + 6, gz + 6
    amp = torch.as_tensor(_source(c, seed), device=fd.dev).double()
    one = c.get("shot", 0) >= 0
    n = c["ns"] if c["kind"] == "shots" else 1
    who = torch.arange(c["ns"], device=fd.dev)
    if c["kind"] != "shots":
        who = who[c["shot"]:c["shot"] + 1] if one else who
    ent = torch.arange(n, device=fd.dev) if c["kind"] == "shots" else torch.zeros_like(who)

    def inject(f, t, sign):
        a = amp[t].expand(len(who)) if one else amp[t]
        f.index_put_((ent, sx[who], sz[who]), sign * a, accumulate=True)

    nt, nx, nz, nb = c["nt"], fd.rv.shape[1], fd.rv.shape[2], c["nb"] + 6
    cur, prev = fd.zeros(n), fd.zeros(n)
    inject(cur, 0, 1.0)
    rec = [] if not gradient else None
    band = torch.zeros((nx, nz), dtype=torch.bool, device=fd.dev)
    band[nb - 6:nx - nb + 6, nz - nb:nz - nb + 6] = True
    band[nb - 6:nb, 6:nz - nb] = True
    band[nx - nb:nx - nb + 6, 6:nz - nb] = True
    saved = []
    for it in range(nt):
        if gradient:
            saved.append(cur[0][band])
        else:
            rec.append(cur[:, gx, gz])
        fd.step(cur, prev)
        cur, prev = prev, cur
        if it + 1 < nt:
            inject(cur, it + 1, 1.0)
    if not gradient:
        return torch.stack(rec, 1)
    s_cur, s_prev = prev, cur  # p(nt-1), p(nt)
    w = _taper(nt, DT)
    vsrc = torch.as_tensor(_traces(nt, c["nx"], 1, _fm(c["dx"]), DT, seed)[0], device=fd.dev).double()
    g_cur, g_prev, grad = fd.zeros(1), fd.zeros(1), fd.zeros(1)[0]
    g_cur[0].index_put_((gx, gz), vsrc[nt - 1], accumulate=True)
    for it in range(nt - 1, -1, -1):
        if w[it] == 0:
            break
        fd.step(s_cur, s_prev, False)
        inject(s_prev, it, -1.0)
        grad[6:-6, 6:-6] -= (w[it] * s_prev * g_cur)[0, 6:-6, 6:-6]
        fd.step(g_cur, g_prev)
        if it >= 1:
            s_prev[0][band] = saved[it - 1]
            g_prev[0].index_put_((gx, gz), vsrc[it - 1], accumulate=True)
        s_cur, s_prev, g_cur, g_prev = s_prev, s_cur, g_prev, g_cur
    return grad


def _net64(p, r, w, x0, x1, z0, z1):
    """The network's correction on its region; one entry at a time."""
    w = torch.as_tensor(w, device=p.device).double()
    w1, w2, w3 = w[:288].view(9, 2, 16), w[288:2592].view(9, 16, 16), w[2592:].view(9, 16)
    a, b = slice(x0 - 3, x1 + 3), slice(z0 - 3, z1 + 3)
    h = torch.stack([p[a, b], (r * p)[a, b]])
    for m in (w1, w2, w3[:, :, None]):
        n = h.shape[1] - 2, h.shape[2] - 2
        o = sum(m[t].T @ h[:, t // 3:t // 3 + n[0], t % 3:t % 3 + n[1]].reshape(h.shape[0], -1) for t in range(9))
        h = o.reshape(-1, *n) if m.shape[2] == 1 else o.reshape(-1, *n).clamp_min(0)
    return h[0]


def _exact_batch(c, seed):
    coarse = c["kind"] == "coarse"
    groups = _groups(c, 2 * DT if coarse else DT)
    dobs, o, grads, vs = _batch_data(groups, seed), 0, [], []
    for g, ms in zip(groups, _batch_models(c, groups, seed)):
        for v in ms:
            fd = _Fd(v, g.nb + 6, 4 if coarse else 10, g.dscale)
            n, nt, bx = g.ns, g.nt, g.nb + 6
            d = torch.as_tensor(dobs[o:o + n * nt * g.ng], device=fd.dev).double().view(n, nt, g.ng)
            o += n * nt * g.ng
            e = torch.arange(n, device=fd.dev)
            sx = torch.as_tensor(np.asarray(g.sx).astype(np.int64) + bx, device=fd.dev)
            amp = _ricker(nt, g.fm, g.dt).astype(np.float64)
            w = 4 * _taper(nt, g.dt)
            first = min(it for it in range(4, nt) if w[it] and it % 4 == 0)
            cur, prev = fd.zeros(n), fd.zeros(n)
            cur[e, sx, 7] += amp[0]
            rec, snap = [], {}
            region = (bx, g.nxpad - bx, 6, g.nzpad - bx)
            for it in range(nt):
                rec.append(cur[:, bx:bx + g.ng, 6].clone())
                if (it + 1) % 4 == 0 and it + 1 < nt and w[it + 1] and it + 1 >= first:
                    snap[it] = cur.clone()
                fd.step(cur, prev)
                cur, prev = prev, cur
                if it + 1 < nt:
                    cur[e, sx, 7] += amp[it + 1]
                if coarse and (it + 2) % 4 == 0:
                    x0, x1, z0, z1 = region
                    for f in (prev, cur):
                        for q in range(n):
                            f[q, x0:x1, z0:z1] += _net64(f[q], fd.rv[0], _weights(seed), *region)
            res = d - torch.stack(rec, 1)
            v = torch.zeros_like(res)
            v[:, 2:nt - 2] = -(res[:, :nt - 4] + res[:, 4:]) / 12 + 4 / 3 * (res[:, 1:nt - 3] + res[:, 3:nt - 1]) - \
                2.5 * res[:, 2:nt - 2]
            vs.append(v.flatten())
            cur, prev, grad = fd.zeros(n), fd.zeros(n), fd.zeros(1)[0]
            cur[:, bx:bx + g.ng, 6] += v[:, nt - 1]
            for it in range(nt - 1, first - 1, -1):
                if it % 4 == 0 and w[it]:
                    grad[6:-6, 6:-6] -= w[it] * (snap[it - 1] * cur).sum(0)[6:-6, 6:-6]
                fd.step(cur, prev)
                cur, prev = prev, cur
                if it - 1 >= first:
                    cur[:, bx:bx + g.ng, 6] += v[:, it - 1]
            grads.append(grad.flatten())
    out = {"gradient": torch.cat(grads).cpu()}
    return {**out, "vsrc": torch.cat(vs).cpu()} if coarse else out


def exact(case, seed):
    c, k = dict(case), case["kind"]
    if k == "step":
        prev, cur = _wave(c, seed)
        fd = _Fd(_padded(_model(c["nx"], c["nz"], seed), c["nb"], 10.0, DT), c["nb"] + 6)
        p, q = (torch.as_tensor(a, device=fd.dev).double()[None] for a in (prev, cur))
        u2 = torch.zeros_like(p)
        u2[:, 5:-5, 5:-5] = fd.step(q, p, c["damped"])
        return {"next": p[0].cpu(), "u2": u2[0].cpu()}
    if k == "forward":
        return _exact_shots(c, seed)[0].cpu()
    if k == "shots":
        return _exact_shots(c, seed).cpu()
    if k == "gradient":
        return _exact_shots(c, seed, True).cpu()
    if k in ("batch", "coarse"):
        return _exact_batch(c, seed)
    return None  # a line search, an ensemble's eigenvectors and Adam's signs: whole calls, not single results
