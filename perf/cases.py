"""The work a user of this library has it do, as cases that can be timed.

Every case goes through a public entry point of mumfim_amd:

  solve      one batch of RVE solves under given deformation gradients
  tangent    stress and 6x6 tangent of a batch (run_with_tangent)
  fe2        one macro Newton iteration through the FE2 record adapter
  predict    the learned surrogate: stress, spread and, where asked, Jacobian
  fit        training of the surrogate ensemble

Networks are random k-nearest-neighbour graphs in the unit cube, as the
repository's generator makes them, built here from the seed.  `exact` solves
the same cases in plain float64 torch.
"""
import math

import numpy as np
import torch

import mumfim_amd as mf

DEV = "cuda"


# ---- cases -----------------------------------------------------------------
def _solve(name, precision, law, n_rve, lo, hi, steps, amp, host=False):
    return {"name": name, "kind": "solve", "precision": precision, "law": law, "n_rve": n_rve,
            "nodes_min": lo, "nodes_max": hi, "steps": steps, "amp": amp, "host": host}


def _tangent(name, scheme, n_rve, lo, hi, steps):
    return {"name": name, "kind": "tangent", "scheme": scheme, "law": "toe", "n_rve": n_rve,
            "nodes_min": lo, "nodes_max": hi, "steps": steps, "amp": 0.05}


def _predict(name, n, members, jacobian):
    return {"name": name, "kind": "predict", "n": n, "members": members, "jacobian": jacobian}


def listed():
    return [
        # One integration point through host buffers: the smallest call, all
        # latency (a material-point driver, or one element being debugged).
        _solve("point_fp32", "fp32", "linear", 1, 180, 180, 500, 0.05, host=True),
        # One macro Newton iteration of a small FE2 problem: a few elements'
        # integration points, the reference's own scheme (relaxed in FP64 until
        # the residual is small, forward-difference tangent), networks of the
        # golden network's size, radius and stiffness.
        {"name": "fe2_newton", "kind": "fe2", "n_rve": 12, "nodes_min": 200, "nodes_max": 400,
         "amp": 0.002},
        # FP64 stress of a whole macro mesh of ordinary linear networks.
        _solve("mesh_fp64", "fp64", "linear", 1024, 500, 500, 1000, 0.05),
        # FP64 over ragged networks of both fiber laws.
        _solve("ragged_fp64", "fp64", "toe", 257, 200, 4000, 600, 0.1),
        # The headline batch: 4096 linear 500-node RVEs, 5000 steps, FP32
        # with compensated positions.
        _solve("headline_fp32", "fp32", "linear", 4096, 500, 500, 5000, 0.05),
        # FP32 over 200 to 4000 nodes, half the fibers on the toe law.
        _solve("ragged_fp32", "fp32", "toe", 1500, 200, 4000, 2000, 0.1),
        # Stress and tangent, FP64 central differences (13 solves per RVE).
        _tangent("tangent_fp64", "central", 64, 1000, 2000, 800),
        # Stress and tangent, FP32 tangent-linear solves (6 per RVE).
        _tangent("tangent_fp32", "linear", 256, 1000, 2000, 800),
        # Surrogate for a small mesh: one call, stress and tangent.
        _predict("surrogate_small", 777, 4, True),
        # Surrogate stress of a large mesh.
        _predict("surrogate_stress", 1 << 20, 4, False),
        # Surrogate stress and tangent of a mesh.
        _predict("surrogate_tangent", 150001, 4, True),
        # Two epochs of ensemble training (the default mini-batch).
        {"name": "train", "kind": "fit", "n": 131072, "members": 4, "batch": 4096, "epochs": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "tangent", "fe2", "predict", "predict", "fit"])
    if kind == "solve":
        precision = rng.choice(["fp32", "fp32", "fp64"])
        law = rng.choice(["linear", "toe"])
        lo = _log(rng, 120, 2500)
        hi = rng.choice([lo, min(4000, int(lo * rng.uniform(1.2, 3.0)))])
        steps = _log(rng, 200, 2000)
        most = 3.0e8 if precision == "fp32" else 5.0e7  # node-steps of a batch
        top = max(2, min(2048, int(most / steps / (0.5 * (lo + hi)))))
        n = _log(rng, 1, top)
        c = _solve("", precision, law, n, lo, hi, steps, rng.choice([0.05, 0.1]), n <= 16)
    elif kind == "tangent":
        scheme = rng.choice(["central", "linear"])
        lo = _log(rng, 200, 1500)
        hi = int(lo * rng.uniform(1.0, 1.6))
        steps = _log(rng, 200, 1000)
        most = 4.0e6 if scheme == "central" else 5.0e7
        c = _tangent("", scheme, _log(rng, 1, max(2, min(512, int(most / steps / lo)))), lo, hi,
                     steps)
        c["law"] = rng.choice(["linear", "toe"])
    elif kind == "fe2":
        lo = _log(rng, 150, 400)
        c = {"kind": "fe2", "n_rve": rng.randint(1, 12), "nodes_min": lo,
             "nodes_max": int(lo * rng.uniform(1.0, 1.5)), "amp": 0.002}
    elif kind == "predict":
        jac = rng.random() < 0.5
        c = _predict("", _log(rng, 1, 200000 if jac else 1 << 20), rng.randint(1, 8), jac)
    else:
        batch = 256 * rng.randint(1, 32)
        c = {"kind": "fit", "n": batch * rng.randint(4, 16) + rng.randint(0, 255),
             "members": rng.randint(1, 6), "batch": batch, "epochs": rng.randint(1, 2)}
    c.pop("name", None)
    return c


def work(case):
    if case["kind"] == "predict":
        planes = 7 if case["jacobian"] else 1
        layer = 2 * (10 * 256 + 2 * 256 * 256 + 256 * 6)
        out = 12 + (36 if case["jacobian"] else 0)
        return {"bytes": 4.0 * case["n"] * (10 + out) + 543768.0 * case["members"],
                "flops": float(case["n"]) * case["members"] * layer * planes}
    if case["kind"] == "fit":
        steps = case["epochs"] * (case["n"] // case["batch"])
        samples = float(steps) * case["batch"] * case["members"]
        # forward, input gradients and weight gradients: three products
        return {"bytes": samples * 64 + steps * case["members"] * 135942.0 * 24,
                "flops": samples * 6 * (10 * 256 + 2 * 256 * 256 + 256 * 6)}
    nodes = 0.5 * (case["nodes_min"] + case["nodes_max"])
    if case["nodes_max"] > 2 * case["nodes_min"]:  # sizes spread over their logarithm
        nodes = ((case["nodes_max"] - case["nodes_min"])
                 / math.log(case["nodes_max"] / case["nodes_min"]))
    fibers = 2.49 * nodes
    if case["kind"] == "fe2":
        solves, steps = 7, 3000  # the steps to the tolerance vary
    else:
        solves = 1
        if case["kind"] == "tangent":
            solves = 13 if case["scheme"] == "central" else 7
        steps = case["steps"]
    per_fiber = 60 if case.get("law") == "toe" else 27
    flops = case["n_rve"] * solves * steps * (per_fiber * fibers + 24 * nodes)
    size = case["n_rve"] * (24 * nodes + 12 * fibers + 72 + 48 + (288 if solves > 1 else 0))
    return {"bytes": float(size), "flops": float(flops)}


# ---- networks --------------------------------------------------------------
def _neighbours(X, k):
    """Indices of the k nearest other nodes of every node; X (r, n, 3)."""
    r, n, _ = X.shape
    out = torch.empty(r, n, k, dtype=torch.int64, device=X.device)
    step = max(1, int(1.0e8 // (n * n)))
    for a in range(0, r, step):
        x = X[a:a + step]
        d2 = sum((x[:, :, None, i] - x[:, None, :, i]) ** 2 for i in range(3))
        d2.diagonal(dim1=1, dim2=2).fill_(math.inf)
        out[a:a + step] = d2.topk(k, dim=2, largest=False).indices
    return out


def _networks(case, seed):
    """The batch's networks: uniform nodes, k-nearest-neighbour fibers, the
    nodes within 0.02 of the cube's faces prescribed."""
    rng = np.random.default_rng([int(seed), 17])
    R, lo, hi = case["n_rve"], case["nodes_min"], case["nodes_max"]
    if hi > 2 * lo:
        sizes = np.rint(np.exp(rng.uniform(math.log(lo), math.log(hi), R))).astype(np.int64)
    else:
        sizes = rng.integers(lo, hi + 1, R)
    coords = [c for c in np.split(rng.uniform(-0.5, 0.5, (int(sizes.sum()), 3)),
                                  np.cumsum(sizes)[:-1])]
    order = np.argsort(sizes, kind="stable")
    keys = []
    for a in range(0, R, 64):
        grp = order[a:a + 64]
        top = int(sizes[grp].max())
        pad = np.empty((len(grp), top, 3))
        pad[:] = 10.0 + 10.0 * np.arange(top)[None, :, None]  # far from every node
        for i, r in enumerate(grp):
            pad[i, :sizes[r]] = coords[r]
        nb = _neighbours(torch.from_numpy(pad).to(DEV), 4)
        me = torch.arange(top, device=DEV)[None, :, None].expand_as(nb)
        real = (torch.arange(top, device=DEV)[None, :]
                < torch.from_numpy(sizes[grp]).to(DEV)[:, None])[:, :, None].expand_as(nb)
        who = torch.from_numpy(grp).to(DEV)[:, None, None].expand_as(nb)
        key = (who << 32) | (torch.minimum(me, nb) << 16) | torch.maximum(me, nb)
        keys.append(torch.unique(key[real]))
    key = torch.cat(keys).sort().values.cpu().numpy()
    ends = np.searchsorted(key >> 32, np.arange(1, R))
    fibers = np.split(np.stack([(key >> 16) & 0xFFFF, key & 0xFFFF], 1).astype(np.int32), ends)
    if case["kind"] == "fe2":
        rx = [mf.Reaction(mf.MF_REACTION_LINEAR, 5.0e-5, 1.0e8, 1000.0)]
    else:
        rx = [mf.Reaction(mf.MF_REACTION_LINEAR, 3.5e-8, 4.32e7, 1000.0),
              mf.Reaction(mf.MF_REACTION_NONLINEAR, 3.5e-8, 4.32e7, 1000.0, 1.2, 1.05, 1.0)]
    toe = case.get("law") == "toe"
    which = np.split((rng.random(len(key)) < (0.5 if toe else 0.0)).astype(np.int32), ends)
    nets = []
    for r in range(R):
        near = np.flatnonzero(0.5 - np.abs(coords[r]).max(1) <= 0.02).astype(np.int32)
        nets.append(mf.Network(coords[r], fibers[r], near, rx, which[r]))
    return nets


def _gradients(n, amp, seed):
    u = np.random.default_rng([int(seed), 23]).uniform(-amp, amp, (n, 3, 3))
    return np.eye(3)[None] + 0.5 * (u + u.transpose(0, 2, 1))


# ---- surrogate inputs ------------------------------------------------------
WIDTHS = (10, 256, 256, 256, 6)


def _weights(rng):
    w = []
    for i, o in zip(WIDTHS[:-1], WIDTHS[1:]):
        b = 1.0 / math.sqrt(i)
        w += [rng.uniform(-b, b, (o, i)), rng.uniform(-b, b, o)]
    return [a.astype(np.float32) for a in w]


def _points(case, seed):
    """Inputs (strain, node count, fibers per volume, mean length, nonlinear
    share), the weights of every member and the normalisation."""
    rng = np.random.default_rng([int(seed), 31])
    n = case["n"]
    X = np.empty((n, 10), np.float32)
    X[:, :6] = rng.uniform(-0.1, 0.1, (n, 6))
    X[:, 6] = rng.integers(200, 4001, n)
    X[:, 7] = 2.49 * X[:, 6] * rng.uniform(0.97, 1.03, n)
    X[:, 8] = 0.6 * X[:, 6] ** (-1 / 3) * rng.uniform(0.97, 1.03, n)
    X[:, 9] = 0.5 * rng.integers(0, 2, n)
    lo = np.array([-0.1] * 6 + [200, 498, 0.038, 0], np.float32)
    hi = np.array([0.1] * 6 + [4000, 9960, 0.103, 0.5], np.float32)
    norm = [0.5 * (lo + hi), 0.29 * (hi - lo),
            np.zeros(6, np.float32), np.full(6, 3.0e-9, np.float32)]
    weights = [_weights(rng) for _ in range(case["members"])]
    return X, weights, [a.astype(np.float32) for a in norm], rng


def _targets(X, rng):
    """Stress-like targets: a quadratic in the strain, stiffer with fibers."""
    e = X[:, :6].astype(np.float64)
    a, b = rng.normal(size=(6, 6)), rng.normal(size=(6, 6, 6))
    y = e @ a + 4.0 * np.einsum("ni,nj,kij->nk", e, e, b, optimize=True)
    y *= (1.0 + X[:, 7:8] / 1.0e4) * 2.0e-8
    return (y + rng.normal(size=y.shape) * 3.0e-10).astype(np.float32)


# ---- prepare and run -------------------------------------------------------
def _params(case):
    p = dict(mode=mf.MF_MODE_RAMP, n_steps=case["steps"],
             reaction_policy=mf.MF_REACT_PER_FIBER)
    if case["kind"] == "solve":
        p["precision"] = mf.MF_PREC_FP32C if case["precision"] == "fp32" else mf.MF_PREC_FP64
    elif case["scheme"] == "central":
        p.update(tangent_scheme=mf.MF_TANGENT_CENTRAL, fd_step=1e-6)
    else:
        p.update(precision=mf.MF_PREC_FP32C, tangent_precision=mf.MF_PREC_FP32C,
                 tangent_scheme=mf.MF_TANGENT_LINEAR)
    return mf.default_params(**p)


FO_RADIUS, FO_FRACTION = 5.0e-5, 0.003
# an increment of 0.2% strain relaxes to about a hundredth of its first forces
FO_TOLERANCE, FO_STEPS = 1.0e-5, 20000


def prepare(case, seed):
    s = {"case": case}
    kind = case["kind"]
    if kind in ("predict", "fit"):
        X, weights, norm, rng = _points(case, seed)
        m = mf.SurrogateMLP(n_members=case["members"], seed=1)
        m.set_normalization(*norm)
        for i, w in enumerate(weights):
            m.set_weights(i, np.concatenate([a.ravel() for a in w]))
        s.update(m=m, X=torch.from_numpy(X).to(DEV))
        if kind == "fit":
            s.update(Y=torch.from_numpy(_targets(X, rng)).to(DEV), seed=int(seed) % 1000 + 1)
        else:
            n = case["n"]
            s.update(Y=torch.empty(n, 6, device=DEV), S=torch.empty(n, 6, device=DEV),
                     J=torch.empty(n, 6, 6, device=DEV) if case["jacobian"] else None)
        return s
    nets = _networks(case, seed)
    F = _gradients(case["n_rve"], case["amp"], seed)
    if kind == "fe2":
        n = len(nets)
        hdrs = np.zeros((n, 7), np.int32)
        hdrs[:, 0] = mf.MF_FO_FIBER_ONLY
        prms = np.zeros((n, 8))
        prms[:, 0], prms[:, 1], prms[:, 5:8] = FO_RADIUS, FO_FRACTION, [0.0, 0.6, 0.8]
        slvr = np.zeros((n, 8))
        slvr[:, 5], slvr[:, 6] = 100.0, 0.8
        sint = np.zeros((n, 10), np.int32)
        sint[:, 0] = mf.MF_FO_SOLVER_EXPLICIT
        s["fo"] = mf.MultiscaleRVEAdapter(nets, hdrs, prms, slvr, sint,
                                          mf.default_params(tolerance=FO_TOLERANCE, max_steps=FO_STEPS))
    else:
        s["g"] = mf.BatchedFiberRVEAnalysisExplicit(nets, _params(case))
    # committed increments are taken back by the next pass: a load cycle
    s.update(F=F, back=np.linalg.inv(F), turn=0)
    if kind == "solve" and not case["host"]:
        n = case["n_rve"]
        s["F_dev"] = torch.from_numpy(F.reshape(n, 9)).to(DEV)
        s["sigma"] = torch.empty(n, 6, dtype=torch.float64, device=DEV)
        s["status"] = torch.empty(n, dtype=torch.int32, device=DEV)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "predict":
        state["m"].predict_device(state["X"], case["n"], state["Y"], state["J"], state["S"])
        out = {"y": state["Y"], "spread": state["S"]}
        return out if state["J"] is None else dict(out, J=state["J"])
    if kind == "fit":
        m = state["m"]
        loss = m.fit(state["X"], state["Y"], case["n"], epochs=case["epochs"],
                     batch=case["batch"], lr=1e-3, lr_final=1e-5, seed=state["seed"])
        return {"loss": loss, "weights": [m.get_weights(i) for i in range(case["members"])]}
    if kind == "solve":
        if case["host"]:
            sigma, status = state["g"].run(state["F"], update_coords=False, return_status=True)
            return {"sigma": sigma, "status": status}
        state["g"].run_device(state["F_dev"], state["sigma"], status_dev=state["status"])
        return {"sigma": state["sigma"], "status": state["status"]}
    F = state["back"] if state["turn"] else state["F"]
    state["turn"] ^= 1
    if kind == "fe2":
        results, status = state["fo"].run(F, return_status=True)
        return {"results": results, "status": status}
    sigma, C, status = state["g"].run_with_tangent(F, return_status=True)
    return {"sigma": sigma, "C": C, "status": status}


# ---- exact: plain float64 torch ---------------------------------------------
class _Flat:
    """A list of networks as one flat graph; node arrays are (3, nodes)."""

    def __init__(self, nets):
        off = np.concatenate([[0], np.cumsum([len(n.coords) for n in nets])])
        fib = np.concatenate([n.fibers.astype(np.int64) + off[i] for i, n in enumerate(nets)])
        law = np.concatenate([np.asarray(n.fiber_reaction) for n in nets])
        bnd = np.concatenate([n.boundary.astype(np.int64) + off[i] for i, n in enumerate(nets)])
        self.R = len(nets)
        self.X = torch.from_numpy(np.concatenate([n.coords for n in nets]).T.copy()).to(DEV)
        self.a, self.b = torch.from_numpy(fib.T.copy()).to(DEV)
        self.toe = torch.from_numpy(law).to(DEV) == 1
        self.any_toe = bool((law == 1).any())
        d = self.X[:, self.b] - self.X[:, self.a]
        self.l0 = (d * d).sum(0).sqrt()
        self.rve = torch.from_numpy(np.repeat(np.arange(self.R), np.diff(off))).to(DEV)
        self.fibers_rve = self.rve[self.a]
        self.fixed = torch.zeros(self.X.shape[1], dtype=torch.bool, device=DEV)
        self.fixed[torch.from_numpy(bnd).to(DEV)] = True
        q = nets[0].reactions[0]
        self.EA, self.c = q.E * math.pi * q.radius ** 2, math.sqrt(q.E / q.density)
        half = 0.5 * q.density * math.pi * q.radius ** 2 * self.l0
        self.mass = torch.zeros_like(self.X[0]).index_add_(0, self.a, half)
        self.mass.index_add_(0, self.b, half)
        self.im = torch.where(self.fixed, 0.0, 1.0 / self.mass)
        if self.any_toe:
            t = nets[0].reactions[1]
            self.B, self.alpha = t.B, self.EA / t.B
            self.ends = [(x, self.alpha * ((1 + x * x * t.B) * math.exp(0.5 * t.B * (x * x - 1)) - 1),
                          self.alpha * x * math.expm1(0.5 * t.B * (x * x - 1)))
                         for x in (t.length_ratio_trns, t.cmp_ratio_trns)]

    def tension(self, e, rate):
        """t = f / l from e = lambda^2 - 1, and dt/de if asked."""
        k = 0.5 * self.EA / self.l0
        t, dt = k * e, k if rate else None
        if self.any_toe:
            lam = (1.0 + e).sqrt()
            toe = (self.alpha / self.l0) * torch.expm1(0.5 * self.B * e)
            dtoe = k * torch.exp(0.5 * self.B * e) if rate else None
            for (x, K, b), out in zip(self.ends, (lam > self.ends[0][0], lam < self.ends[1][0])):
                toe = torch.where(out, (K - (K * x - b) / lam) / self.l0, toe)
                if rate:
                    dtoe = torch.where(out, 0.5 * (K * x - b) / (lam ** 3 * self.l0), dtoe)
            t = torch.where(self.toe, toe, t)
            dt = torch.where(self.toe, dtoe, dt) if rate else None
        return t, dt

    def scatter(self, e):
        """Internal force of the nodes from the fibers' force vectors."""
        f = torch.zeros_like(self.X)
        for k in range(3):
            f[k].index_add_(0, self.b, e[k])
            f[k].index_add_(0, self.a, e[k], alpha=-1)
        return f

    def forces(self, x, dx=None, shortest=False):
        """Internal force of every node (and its derivative), and the shortest
        fiber of every RVE with its derivative."""
        d = x.index_select(1, self.b) - x.index_select(1, self.a)
        l2 = (d * d).sum(0)
        t, dt = self.tension(l2 / self.l0 ** 2 - 1.0, dx is not None)
        f = self.scatter(d * t)
        df = dl2 = None
        if dx is not None:
            dd = dx.index_select(1, self.b) - dx.index_select(1, self.a)
            dl2 = 2.0 * (d * dd).sum(0)
            df = self.scatter(dd * t + d * (dt * dl2 / self.l0 ** 2))
        lmin = dlmin = None
        if shortest:
            far = torch.full((self.R,), 1e300, dtype=torch.float64, device=DEV)
            l = l2.sqrt()
            lmin = far.scatter_reduce(0, self.fibers_rve, l, "amin")
            if dx is not None:
                M = len(l)
                mine = torch.where(l == lmin[self.fibers_rve], torch.arange(M, device=DEV), M)
                at = torch.full((self.R,), M, device=DEV).scatter_reduce(
                    0, self.fibers_rve, mine, "amin")
                dlmin = dl2[at] / (2.0 * lmin)
        return f, df, lmin, dlmin

    def stress(self, x, f, V):
        p = torch.where(self.fixed, x, 0.0)
        v = torch.stack([p[0] * f[0], p[1] * f[1], p[2] * f[2],
                         0.5 * (p[1] * f[2] + p[2] * f[1]),
                         0.5 * (p[0] * f[2] + p[2] * f[0]),
                         0.5 * (p[0] * f[1] + p[1] * f[0])], 1)
        out = torch.zeros(self.R, 6, dtype=torch.float64, device=DEV)
        return out.index_add_(0, self.rve, v) / V[:, None]


def _affine(g, A, x):
    B = A[g.rve]
    return torch.stack([B[:, i, 0] * x[0] + B[:, i, 1] * x[1] + B[:, i, 2] * x[2]
                        for i in range(3)])


def _ramp(g, F, V, steps, G=None):
    """Stress after a ramp of `steps` steps from the reference configuration
    (and its derivative along dF = G)."""
    eye = torch.eye(3, dtype=torch.float64, device=DEV)
    inc = _affine(g, F - eye, g.X)
    x, v = g.X.clone(), torch.zeros_like(g.X)
    dinc = _affine(g, G, g.X) if G is not None else None
    dx, dv = (torch.zeros_like(x), torch.zeros_like(x)) if G is not None else (None, None)
    f, df, lmin, dlmin = g.forces(x, dx, True)
    f = -f
    df = -df if G is not None else None
    eta = 100.0 * g.mass
    dh = None
    for k in range(steps):
        if k == 0 or (k - 1) % 100 == 0:  # the step follows the last refresh
            h = (0.4 * lmin / g.c)[g.rve]
            dh = (0.4 * dlmin / g.c)[g.rve] if G is not None else None
            him = h * g.im
        if G is not None:
            dv = dv + (dh * f + h * df) * g.im
        v = v + him * f
        a = (k + 1) / steps
        if G is not None:
            dx = torch.where(g.fixed, a * dinc, dx + 2.0 * (dh * v + h * dv))
        x = torch.where(g.fixed, g.X + a * inc, x + 2.0 * h * v)
        fi, dfi, lm, dlm = g.forces(x, dx, k % 100 == 0)
        if lm is not None:
            lmin, dlmin = lm, dlm
        f = -fi - eta * v
        if G is not None:
            df = -dfi - eta * dv
            dv = dv + (dh * f + h * df) * g.im
        v = v + him * f
    s = g.stress(x, fi, V)
    if G is None:
        return s
    return s, g.stress(dx, fi, V) + g.stress(x, dfi, V)


def _relax(g, F, x, u, V, tol, most):
    """The reference loop from coordinates x and displacements u: the affine
    guess on every node, damped steps until the residual is small."""
    eye = torch.eye(3, dtype=torch.float64, device=DEV)
    x = g.X + (_affine(g, F - eye, x) + u)
    v = torch.zeros_like(x)
    fi, _, lmin, _ = g.forces(x, None, True)
    f, eta = -fi, 100.0 * g.mass
    end, fend = x.clone(), fi.clone()
    done = torch.zeros(g.R, dtype=torch.bool, device=DEV)
    for k in range(most):
        h = (0.4 * lmin / g.c)[g.rve]
        v = v + h * f * g.im
        x = torch.where(g.fixed, x, x + 2.0 * h * v)
        fi, _, lm, _ = g.forces(x, None, k % 100 == 0)
        f = -fi - eta * v
        v = v + h * f * g.im
        if lm is not None:
            lmin = lm
            free = torch.where(g.fixed, 0.0, fi)
            res = torch.zeros(g.R, dtype=torch.float64, device=DEV).index_add_(
                0, g.rve, (free * free).sum(0)).sqrt()
            new = ~(res > tol) & ~done
            pick = new[g.rve]
            end, fend = torch.where(pick, x, end), torch.where(pick, fi, fend)
            done |= new
            if bool(done.all()):
                break
    late = ~done[g.rve]
    end, fend = torch.where(late, x, end), torch.where(late, fi, fend)
    return g.stress(end, fend, V), end


def _almansi(i, h):
    D = math.sqrt(1.0 / (1 - 2 * h))
    a, b = math.sqrt((1 + h) / (1 - h * h)), math.sqrt((1 - h) / (1 - h * h))
    P = np.eye(3)
    if i < 3:
        P[i, i] = D
    else:
        j, k = ((1, 2), (0, 2), (0, 1))[i - 3]
        P[j, j] = P[k, k] = 0.5 * (a + b)
        P[j, k] = P[k, j] = 0.5 * (a - b)
    return P


def _rate(i):
    E = np.zeros((3, 3))
    if i < 3:
        E[i, i] = 1.0
    else:
        j, k = ((1, 2), (0, 2), (0, 1))[i - 3]
        E[j, k] = E[k, j] = 0.5
    return E


def _exact_predict(case, seed):
    X, weights, norm, _ = _points(case, seed)
    mean, std, omean, ostd = [torch.from_numpy(a).to(DEV).double() for a in norm]
    x = (torch.from_numpy(X).to(DEV).double() - mean) / std
    seeds = torch.eye(10, dtype=torch.float64, device=DEV)[:6]
    ys, js = [], []
    for w in weights:
        w = [torch.from_numpy(a).to(DEV).double() for a in w]
        a = x
        t = [s.expand_as(x) for s in seeds] if case["jacobian"] else []
        for i in range(0, 8, 2):
            z = a @ w[i].T + w[i + 1]
            t = [p @ w[i].T for p in t]
            if i == 6:
                a = z
                break
            sg = torch.sigmoid(z)
            t = [p * (sg * (1 + z * (1 - sg))) for p in t]
            a = z * sg
        ys.append(a)
        js.append(torch.stack(t, 2) if t else None)
    y = torch.stack(ys)
    out = {"y": y.mean(0) * ostd + omean,
           "spread": y.std(0, unbiased=False) * ostd if len(ys) > 1 else None}
    if case["jacobian"]:
        out["J"] = torch.stack(js).mean(0) * ostd[:, None] / std[:6]
    return out


def _shuffled(n, seed, stream):
    """A Fisher-Yates shuffle of 0..n-1 by SplitMix64 (seed, stream)."""
    u = np.uint64
    gold = 0x9E3779B97F4A7C15

    def mix(z):
        z = (z ^ (z >> u(30))) * u(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> u(27))) * u(0x94D049BB133111EB)
        return z ^ (z >> u(31))

    with np.errstate(over="ignore"):
        start = mix((u(seed) ^ mix(u(stream) + u(gold))) + u(gold))
        draws = mix(start + np.arange(1, n, dtype=u) * u(gold))
    at = (draws % np.arange(n, 1, -1, dtype=u)).tolist()
    p = list(range(n))
    for i, j in zip(range(n - 1, 0, -1), at):
        p[i], p[j] = p[j], p[i]
    return np.array(p)


def _exact_fit(case, seed):
    X, weights, norm, rng = _points(case, seed)
    Y = _targets(X, rng)
    mean, std, omean, ostd = [torch.from_numpy(a).to(DEV).double() for a in norm]
    x = (torch.from_numpy(X).to(DEV).double() - mean) / std
    y = (torch.from_numpy(Y).to(DEV).double() - omean) / ostd
    n, bt, epochs, K = case["n"], case["batch"], case["epochs"], case["members"]
    steps = n // bt
    losses = np.zeros((epochs, K))
    out = []
    for m in range(K):
        w = [torch.from_numpy(a).to(DEV).double().requires_grad_() for a in weights[m]]
        opt = torch.optim.Adam(w, lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
        it = 0
        for ep in range(epochs):
            p = torch.from_numpy(_shuffled(n, int(seed) % 1000 + 1, ep * K + m)).to(DEV)
            for s in range(steps):
                frac = it / (steps * epochs - 1) if steps * epochs > 1 else 1.0
                opt.param_groups[0]["lr"] = 1e-5 + 0.5 * (1e-3 - 1e-5) * (1 + math.cos(math.pi * frac))
                rows = p[s * bt:(s + 1) * bt]
                a = x[rows]
                for i in range(0, 6, 2):
                    a = torch.nn.functional.silu(a @ w[i].T + w[i + 1])
                loss = ((a @ w[6].T + w[7] - y[rows]) ** 2).mean()
                opt.zero_grad()
                loss.backward()
                opt.step()
                losses[ep, m] += float(loss.detach()) / steps
                it += 1
        out.append(torch.cat([a.detach().reshape(-1) for a in w]))
    return {"loss": losses, "weights": out}


def exact(case, seed):
    kind = case["kind"]
    if kind == "predict":
        return _exact_predict(case, seed)
    if kind == "fit":
        return _exact_fit(case, seed)
    nets = _networks(case, seed)
    F = torch.from_numpy(_gradients(case["n_rve"], case["amp"], seed)).to(DEV)
    one = torch.ones(len(nets), dtype=torch.float64, device=DEV)
    if kind == "solve":
        return {"sigma": _ramp(_Flat(nets), F, one, case["steps"]), "status": None}
    V = torch.linalg.det(F)
    if kind == "tangent":
        if case["scheme"] == "central":
            h = 1e-6
            P = [np.eye(3)] + [_almansi(i, s * h) for i in range(6) for s in (1, -1)]
            P = torch.from_numpy(np.stack(P)).to(DEV)
            g = _Flat([n for n in nets for _ in range(13)])
            A = (P[None] @ F[:, None]).reshape(-1, 3, 3)
            s = _ramp(g, A, V.repeat_interleave(13), case["steps"]).reshape(-1, 13, 6)
            C = ((s[:, 1::2] - s[:, 2::2]) / (2 * h)).transpose(1, 2)
            return {"sigma": s[:, 0], "C": C, "status": None}
        E = torch.from_numpy(np.stack([_rate(i) for i in range(6)])).to(DEV)
        g = _Flat([n for n in nets for _ in range(6)])
        G = (E[None] @ F[:, None]).reshape(-1, 3, 3)
        s, ds = _ramp(g, F.repeat_interleave(6, 0), V.repeat_interleave(6), case["steps"], G)
        return {"sigma": s.reshape(-1, 6, 6)[:, 0], "C": ds.reshape(-1, 6, 6).transpose(1, 2),
                "status": None}
    # the reference's sequence: the update run, then six trials, each from the
    # coordinates the last one left and the committed displacements
    g = _Flat(nets)
    length = torch.zeros(g.R, dtype=torch.float64, device=DEV).index_add_(
        0, g.fibers_rve, g.l0)
    V = V * (length * (math.pi * FO_RADIUS ** 2 / FO_FRACTION))
    s0, x = _relax(g, F, g.X, torch.zeros_like(g.X), V, FO_TOLERANCE, FO_STEPS)
    u, h, cols = x - g.X, 1e-5, []
    for i in range(6):
        P = torch.from_numpy(_almansi(i, h)).to(DEV).expand(g.R, 3, 3)
        s, x = _relax(g, P, x, u, V, FO_TOLERANCE, FO_STEPS)
        cols.append((s - s0) / h)
    C = torch.stack(cols, 2).reshape(g.R, 36)
    zero = torch.zeros(g.R, 3, dtype=torch.float64, device=DEV)
    return {"results": torch.cat([s0, zero, C], 1), "status": None}
