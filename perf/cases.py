"""What is timed of this framework, and at which sizes.

A case is one piece of work that a program built on the framework has it do,
through its public entry points: internal steps of the ocean model
(``DeviceModel``), an ensemble cycle (union, forecast, EnKF update), and the
learned closure's trainer (``Trainer``).  ``listed`` gives the fixed cases,
``draw`` one more of the same ranges, ``prepare`` what a program has in hand
before the call, ``run`` one pass, ``work`` the bytes and operations a pass
cannot do without, ``exact`` the result in 64 bits where it is computed by
itself (the trainer; the time step has no independent closed form).

The model's state lives on the GPU and goes on from pass to pass; what a pass
returns are the arrays that such a program reads between its steps (history
output or coupling).
"""
import numpy as np

import myfvcomcode_amd as F
from myfvcomcode_amd import closure, enkf

H = 64
NPARAM = 5 * H + H + H * H + H + 2 * H + 2
MOVES = ("el", "ua", "va", "u", "v", "t1", "s1")   # FVCOM's history fields, and what the EnKF updates


def _step(name, base, nx, ny, kb, steps, precision="fp64", graph=True, learned=False, wind_each=False,
          obc="elevation", river="none", reads="history"):
    c = {"what": "step", "base": base, "nx": nx, "ny": ny, "kb": kb, "steps": steps, "precision": precision,
         "graph": graph, "learned": learned, "wind_each": wind_each, "obc": obc, "river": river, "reads": reads}
    return dict(c, name=name) if name else c


def listed():
    return [
        # INTERNAL_STEP as a host model calls it, one call at a time, on the
        # 81x21-node estuary channel, the coupler reading its fields back
        _step("channel_one_step", 0, 81, 21, 11, 1, graph=False, river="specified"),
        # the same channel run from one output to the next: an hour of 50 s steps
        _step("channel_hour", 0, 81, 21, 11, 72, river="specified"),
        # a surge forecast on an odd-sized mesh: new wind at every step,
        # open boundary with every condition, river T/S calculated
        _step("surge_17k", 1, 127, 67, 21, 6, wind_each=True, obc="mixed", river="calculated"),
        # the bench's generator at 1/16 of its mesh (one subdomain of it)
        _step("seamount_62k", 1, 251, 126, 41, 40),
        # one ensemble member in mixed precision
        _step("member_250k_mixed", 3, 501, 251, 21, 40, precision="mixed"),
        # mixed precision with the learned closure
        _step("closure_125k", 1, 355, 178, 41, 40, precision="mixed", learned=True),
        # the bench's mesh, 1,000,000 elements x 40 layers, FP64
        _step("seamount_1m", 1, 1001, 501, 41, 40, reads="surface"),
        # an ensemble cycle: 24 members of 10,000 elements as one union,
        # forecast, EnKF update of every prognostic array
        {"name": "ensemble_cycle", "what": "cycle", "members": 24, "nx": 101, "ny": 51, "kb": 21, "steps": 6,
         "precision": "mixed"},
        # one gradient of the closure's loss over a small odd batch
        {"name": "mlp_grad_1k", "what": "grad", "samples": 20000, "batch": 1000},
        # training steps at the batch the closure is trained with
        {"name": "mlp_train_8k", "what": "train", "samples": 400000, "batch": 8192, "steps": 10},
        # validation pass, FP32
        {"name": "mlp_infer_f32", "what": "infer", "samples": 400000, "mfma": False},
        # the inference form of the time step, BF16 matrix cores
        {"name": "mlp_infer_mfma", "what": "infer", "samples": 1000000, "mfma": True},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["cycle", "grad", "train", "infer"])
    if kind == "step":
        base = rng.choice([0, 1, 1, 3])
        n = _log(rng, 1200, 260000)                      # elements
        nx = max(13, int((n / 2 * rng.uniform(1.0, 3.0)) ** 0.5) | 1)
        ny = max(9, n // (2 * nx))
        kb = rng.choice([4, 6, 9, 11, 17, 21, 21, 26, 31, 41, 41, 48, 64])
        # steps by cost: a few milliseconds to a quarter of a second
        steps = max(1, min(60, int(6e7 / (n * kb + 60000))))
        graph = rng.random() < 0.8
        learned = base != 0 and kb >= 6 and rng.random() < 0.2
        return _step(None, base, nx, ny, kb, steps, rng.choice(["fp64", "fp64", "mixed"]), graph, learned,
                     base != 0 and rng.random() < 0.3, rng.choice(["elevation", "elevation", "mixed"]),
                     rng.choice(["none", "specified", "calculated", "edge"]))
    if kind == "cycle":
        members = rng.randint(2, 40)
        nx = rng.randrange(31, 121, 2)
        return {"what": "cycle", "members": members, "nx": nx, "ny": max(15, nx // 2 + rng.randint(-4, 4)),
                "kb": rng.choice([6, 11, 21]), "steps": rng.randint(1, 8), "precision": rng.choice(["fp64", "mixed"])}
    if kind == "grad":
        return {"what": "grad", "samples": 30000, "batch": _log(rng, 40, 16000)}
    if kind == "train":
        return {"what": "train", "samples": _log(rng, 20000, 600000), "batch": _log(rng, 500, 16384),
                "steps": rng.randint(1, 20)}
    return {"what": "infer", "samples": _log(rng, 1000, 1000000), "mfma": rng.random() < 0.6}


# ------------------------------------------------------------------ inputs
def _waves(rng, x, y, length, terms=12):
    """A smooth random field of unit variance over points (x, y)."""
    f = np.zeros_like(x)
    for _ in range(terms):
        k = 2.0 * np.pi / (length * rng.uniform(0.7, 2.5))
        a = rng.uniform(0.0, 2.0 * np.pi)
        f += np.cos(k * (np.cos(a) * x + np.sin(a) * y) + rng.uniform(0.0, 2.0 * np.pi))
    return f * np.sqrt(2.0 / terms)


_meshes = {}   # host meshes of this process by shape: a program reads its grid once, and starts runs from it


def _mesh(case):
    key = tuple(case[k] for k in ("base", "nx", "ny", "kb", "obc", "river"))
    if key in _meshes:
        return _meshes[key]
    base = case["base"]
    kw = dict(nx=case["nx"], ny=case["ny"], kb=case["kb"], sponge_radius=0.0, river=0, el_pert_std=0.0)
    if base:
        kw.update(wind=0, n_seamounts=max(1, min(20, round(20 * case["nx"] * case["ny"] / 125751))))
    kw["p_river_ts_specified"] = 0 if case["river"] in ("calculated", "edge") else 1
    m = F.Model.build(base, **kw)
    # the sponge along the eastern open boundary (4 km, 0.01)
    xc, lx = m.field("xc"), m.field("vx")[1:].max()
    m.field("cc_sponge")[1:] = 0.01 * np.maximum(0.0, 1.0 - (lx - xc[1:]) / 4000.0)
    if case["obc"] == "mixed":
        nob = m.hdr.iobcn
        m.set_obc_type(np.array([1, 2, 5, 6, 7, 8], np.int32)[np.arange(nob) * 6 // nob])
    mid = (case["ny"] // 2) * case["nx"] + 1
    if case["river"] in ("specified", "calculated"):
        m.set_river(mid, 100.0, 15.0, 0.0)
    elif case["river"] == "edge":
        isbce, nbe = m.field("isbce"), m.field("nbe").reshape(3, -1)
        solid = np.nonzero((isbce == 1) & ((nbe == 0).sum(axis=0) == 1))[0]
        solid = solid[solid > 0]
        m.set_river_edge(int(solid[np.argmin(m.field("xc")[solid])]), 100.0, 15.0, 0.0)
    start = {n: m.field(n).copy() for n in ("el", "t1", "s1")}
    _meshes[key] = (m, start)
    return _meshes[key]


def _wind(rng, m):
    """A wind field of 8 m/s with 2 m/s of variation, UUWIND and VVWIND."""
    x, y = m.field("xc"), m.field("yc")
    a = rng.uniform(0.0, 2.0 * np.pi)
    u = 8.0 * np.cos(a) + 2.0 * _waves(rng, x, y, 50000.0, 4)
    v = 8.0 * np.sin(a) + 2.0 * _waves(rng, x, y, 50000.0, 4)
    u[0] = v[0] = 0.0
    return u, v


def _start_state(rng, m, start, base):
    """The cold start of a run: a perturbed sea level and stratification."""
    for n, a in start.items():
        m.field(n)[:] = a
    x, y = m.field("vx")[1:], m.field("vy")[1:]
    m.field("el")[1:] = 0.05 * _waves(rng, x, y, 20000.0)
    dt, ds = 0.3 * _waves(rng, x, y, 30000.0, 4), 0.2 * _waves(rng, x, y, 30000.0, 4)
    t1, s1 = m.field3("t1"), m.field3("s1")
    for k in range(m.kb - 1):
        t1[k, 1:] += dt
        s1[k, 1:] = np.maximum(0.0, s1[k, 1:] + ds)
    if base:
        u, v = _wind(rng, m)
        for n, w in (("uuwind", u), ("vvwind", v), ("uuwind0", u), ("vvwind0", v)):
            m.field(n)[:] = w
    m.cold_start()


def _samples(case, seed):
    """Closure samples of the ranges that the model's own states have."""
    n = case["samples"]
    rng = np.random.default_rng(seed)
    x = np.zeros((n, 8), np.float32)
    x[:, 0] = rng.normal(0, 2, n)
    x[:, 1] = rng.normal(0, 1, n)
    x[:, 2] = -rng.uniform(0, 1, n)
    x[:, 3] = rng.uniform(0, 2, n)
    x[:, 4] = rng.normal(0, 0.5, n)
    x[:, 5] = 1.0
    y = np.exp(rng.uniform(np.log(1e-5), np.log(1e-1), (n, 2))).astype(np.float32)
    idx = rng.integers(0, n, case.get("batch", 1)).astype(np.int32)
    return x, y, idx


def _params(seed):
    """He-scaled random weights (the network before training)."""
    rng = np.random.default_rng(seed + 77)
    p = np.zeros(NPARAM, np.float32)
    p[:5 * H] = rng.normal(0.0, np.sqrt(2.0 / 5), 5 * H)
    p[6 * H:6 * H + H * H] = rng.normal(0.0, np.sqrt(2.0 / H), H * H)
    o = 7 * H + H * H
    p[o:o + 2 * H] = rng.normal(0.0, np.sqrt(1.0 / H), 2 * H)
    p[o + 2 * H:] = np.log(np.expm1(1e-3))
    return p


def prepare(case, seed):
    what = case["what"]
    if what == "step":
        rng = np.random.default_rng(seed)
        m, start = _mesh(case)
        _start_state(rng, m, start, case["base"])
        dev = F.DeviceModel(m, precision=case["precision"])
        if case["learned"]:
            dev.set_closure(1, closure.load_params())
        winds = None
        if case["wind_each"]:
            winds = [np.concatenate(_wind(rng, m)) for _ in range(8)]
        dev.synchronize()
        return {"case": case, "dev": dev, "model": m, "winds": winds, "at": 0}
    if what == "cycle":
        parts = []
        for j in range(case["members"]):
            rng = np.random.default_rng([seed, j])
            m, start = _mesh(dict(case, base=3, obc="elevation", river="none"))
            _start_state(rng, m, start, 3)
            parts.append(F.Model.union([m])[0])          # the member's own copy
        union, offs = F.Model.union(parts)
        dev = F.DeviceModel(union, precision=case["precision"])
        ens = enkf.Ensemble(union, offs, case["members"])
        n = case["members"]
        q = np.linalg.qr(np.random.default_rng(seed).standard_normal((n, n)))[0]
        c = np.eye(n) - np.ones((n, n)) / n
        # mean kept, anomalies mixed a little and drawn together
        x5 = np.ones((n, n)) / n + 0.995 * c @ (0.98 * np.eye(n) + 0.02 * q) @ c
        dev.synchronize()
        return {"case": case, "dev": dev, "ens": ens, "x5": x5, "parts": parts}
    x, y, idx = _samples(case, seed)
    t = F.Trainer(x, y, bmax=case.get("batch", 1))
    t.set_params(_params(seed))
    return {"case": case, "trainer": t, "idx": idx, "seed": seed}


def run(state):
    case = state["case"]
    what = case["what"]
    if what == "step":
        dev, steps = state["dev"], case["steps"]
        if case["wind_each"]:
            for _ in range(steps):
                dev.set_forcing("wind", state["winds"][state["at"] % 8])
                state["at"] += 1
                if case["graph"]:
                    dev.run(1)
                else:
                    dev.internal_step()
        elif case["graph"]:
            dev.run(steps)
        else:
            for _ in range(steps):
                dev.internal_step()
        return {n: dev.get(n) for n in (MOVES if case["reads"] == "history" else ("el", "ua", "va", "t1", "s1"))}
    if what == "cycle":
        dev, ens = state["dev"], state["ens"]
        dev.run(case["steps"])
        for n in MOVES:
            ens.update(dev, n, state["x5"])
        return {n: dev.get(n) for n in MOVES}
    t = state["trainer"]
    if what == "grad":
        loss, g = t.grad(state["idx"])
        return {"loss": loss, "grad": g}
    if what == "train":
        loss = t.train(case["steps"], batch=case["batch"], seed=state["seed"])
        return {"loss": loss, "params": t.params()}
    return t.infer(0, case["samples"], mfma=case["mfma"])


# ------------------------------------------------------------------ floors
def _sizes(nx, ny, kb, copies=1):
    m, n = nx * ny, 2 * (nx - 1) * (ny - 1)
    return copies * m, copies * n, copies * (n + m), kb


def _step_bytes(m, n, ne, kb, isplit=10):
    """One internal step: the 2-D fields and geometry of every RK stage read
    once and its state written once; then each 3-D array that the step reads
    (nodes: T1 S1 RHO1 and their means, Q2 Q2L KM KH KQ; elements: U V RHO
    RMEAN) and writes (nodes: T1 S1 RHO1 Q2 Q2L L KM KH KQ WTS; elements: U V
    W WW T S RHO KM1) once."""
    stage = 8 * (n * (8 + 16 + 6) + m * 6 + ne * 4) + 4 * (n * 9 + ne * 5)
    stage += 8 * (4 * n + 2 * m)
    return 4 * isplit * stage + 8 * kb * (m * (11 + 10) + n * (4 + 8))


def work(case):
    what = case["what"]
    if what == "step":
        m, n, ne, kb = _sizes(case["nx"], case["ny"], case["kb"])
        b = case["steps"] * _step_bytes(m, n, ne, kb)
        f = case["steps"] * m * (kb - 2) * 2.0 * (NPARAM - 2 * H) if case["learned"] else 0.0
        return {"bytes": b, "flops": f}
    if what == "cycle":
        m, n, ne, kb = _sizes(case["nx"], case["ny"], case["kb"], case["members"])
        values = m * (1 + 2 * kb) + n * (2 + 2 * kb)
        return {"bytes": case["steps"] * _step_bytes(m, n, ne, kb) + 16 * values,
                "flops": 2.0 * values * case["members"]}
    weights = 2.0 * (NPARAM - 2 * H - 2)
    if what == "grad":
        return {"bytes": case["batch"] * 44 + 8 * NPARAM, "flops": 3 * weights * case["batch"]}
    if what == "train":
        return {"bytes": case["steps"] * (case["batch"] * 44 + 32 * NPARAM),
                "flops": 3 * weights * case["batch"] * case["steps"]}
    return {"bytes": case["samples"] * 40 + 4 * NPARAM, "flops": weights * case["samples"]}


# ------------------------------------------------------------------ 64 bits
def _unpack(p):
    o = 6 * H + H * H
    return (p[:5 * H].reshape(H, 5), p[5 * H:6 * H], p[6 * H:o].reshape(H, H), p[o:o + H],
            p[o + H:o + 3 * H].reshape(2, H), p[o + 3 * H:])


def _sig(z):
    return 1.0 / (1.0 + np.exp(-z))


def _forward(p, x):
    w1, b1, w2, b2, w3, b3 = _unpack(p)
    z1 = x @ w1.T + b1
    h1 = z1 * _sig(z1)
    z2 = h1 @ w2.T + b2
    h2 = z2 * _sig(z2)
    o = h2 @ w3.T + b3
    return z1, h1, z2, h2, o, np.where(o > 20.0, o, np.log1p(np.exp(np.minimum(o, 20.0)))) + 1e-7


def _loss_grad(p, x, y):
    w1, b1, w2, b2, w3, b3 = _unpack(p)
    z1, h1, z2, h2, o, k = _forward(p, x)
    r = np.log(k) - np.log(np.maximum(y, 1e-7))
    do = 2.0 * r / k * _sig(o) / len(x)
    s1, s2 = _sig(z1), _sig(z2)
    d2 = (do @ w3) * (s2 * (1.0 + z2 * (1.0 - s2)))
    d1 = (d2 @ w2) * (s1 * (1.0 + z1 * (1.0 - s1)))
    g = [(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), (do.T @ h2).ravel(), do.sum(0)]
    return float(np.mean(np.sum(r * r, axis=1))), np.concatenate(g)


def _adamw(p, x, y, case, seed):
    """fvmlp_train's steps: seeded minibatches (64-bit LCG, high bits) and
    decoupled weight decay on the weight matrices."""
    decay = np.zeros(NPARAM)
    decay[:5 * H] = decay[6 * H:6 * H + H * H] = 1.0
    decay[7 * H + H * H:7 * H + H * H + 2 * H] = 1.0
    lr, wd, b1, b2 = 2e-3, 1e-4, 0.9, 0.999
    mo, ve, mask = np.zeros(NPARAM), np.zeros(NPARAM), (1 << 64) - 1
    st = (seed * 6364136223846793005 + 1442695040888963407) & mask
    loss = 0.0
    for it in range(1, case["steps"] + 1):
        idx = np.empty(case["batch"], np.int64)
        for b in range(case["batch"]):
            st = (st * 6364136223846793005 + 1442695040888963407) & mask
            idx[b] = (st >> 33) % case["samples"]
        loss, g = _loss_grad(p, x[idx], y[idx])
        mo, ve = b1 * mo + (1 - b1) * g, b2 * ve + (1 - b2) * g * g
        p = p - lr * wd * decay * p - lr * (mo / (1 - b1 ** it)) / (np.sqrt(ve / (1 - b2 ** it)) + 1e-8)
    return loss, p


def exact(case, seed):
    if case["what"] in ("step", "cycle"):
        return None
    x, y, idx = _samples(case, seed)
    x, y, p = x[:, :5].astype(np.float64), y.astype(np.float64), _params(seed).astype(np.float64)
    if case["what"] == "grad":
        loss, g = _loss_grad(p, x[idx], y[idx])
        return {"loss": loss, "grad": g}
    if case["what"] == "train":
        loss, p = _adamw(p, x, y, case, seed)
        return {"loss": loss, "params": p}
    return _forward(p, x)[5]
