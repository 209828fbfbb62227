"""Workloads of the cloth library whose time is followed: what each stands for,
its inputs, one pass through the public entry points, and the same results in
64 bits.

A pass is what a program does between two looks at the cloth: a few steps on a
handle it keeps, then the state (or the gradients) read back.  A simulation's
next pass goes on from where the last one ended; a differentiable rollout
starts from its initial state every time, as a training loop does.
"""
import functools
import math

import numpy as np

KS, KD = (50.0, 50.0, 50.0), (-0.25, -0.25, -0.25)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # One displayed frame of the implicit demo: 21x21, StepPhysics with the
        # collider and the Provot pass, state read back for drawing; the solve
        # in one launch, as recommended at demo size.
        {"name": "demo_frame_21", "kind": "physics", "scene": "ie", "nx": 21, "ny": 21, "steps": 1,
         "persistent": True},
        # Ten steps of the Baraff-Witkin demo between two frames: velocity
        # damping, Jacobi-preconditioned solve, relative stopping test.
        {"name": "bw_demo_21", "kind": "physics", "scene": "bw", "nx": 21, "ny": 21, "steps": 10,
         "persistent": False},
        # An ordinary garment panel: odd sides, solve stopped at a relative
        # tolerance, ten steps per frame.
        {"name": "cloth_90x71", "kind": "steps", "nx": 90, "ny": 71, "steps": 10, "tol": "relative"},
        # The headline workload: 512x512, 30 iterations per solve.
        {"name": "cloth_512", "kind": "steps", "nx": 512, "ny": 512, "steps": 20, "tol": "fixed"},
        # The largest cloth: a million vertices, ragged in both directions.
        {"name": "cloth_1023x1001", "kind": "steps", "nx": 1023, "ny": 1001, "steps": 4, "tol": "fixed"},
        # One iteration of a training loop over one cloth: new stiffness, a
        # rollout, a loss on the final positions, gradients.
        {"name": "rollout_128", "kind": "rollout", "nx": 128, "ny": 128, "steps": 24, "every": 8},
        # Many uneven cloths stepped together (sides 16 to 128).
        {"name": "batch_512", "kind": "batch", "cloths": 512, "lo": 16, "hi": 128, "layout": 0, "steps": 100,
         "threads": 1024, "per_thread": 1},
        # The same with gradients (sides 32 to 96).
        {"name": "batch_rollout_64", "kind": "batch_rollout", "cloths": 64, "lo": 32, "hi": 96, "layout": 0,
         "steps": 10, "every": 5, "threads": 1024, "per_thread": 1},
        # The Verlet demo's step on a large cloth with its collider.
        {"name": "verlet_512", "kind": "verlet", "nx": 512, "ny": 512, "steps": 200},
        # One frame of the GPU Verlet demo: one step into the vertex buffer,
        # then wait for it.
        {"name": "vgrid_frame_256", "kind": "vgrid", "nx": 256, "ny": 256, "steps": 1},
        # One frame of the position-based-dynamics demo.
        {"name": "pbd_frame_21", "kind": "pbd", "nx": 21, "ny": 21, "steps": 1},
        # The same constraints on a large cloth.
        {"name": "pbd_512", "kind": "pbd", "nx": 512, "ny": 512, "steps": 10},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["physics", "steps", "steps", "steps", "rollout", "batch", "batch_rollout", "verlet", "vgrid",
                       "pbd"])
    c = {"kind": kind}
    if kind == "physics":  # demo cloths: 12 to 64 a side, one to ten steps a frame
        c.update(scene=rng.choice(["ie", "bw"]), nx=_log_int(rng, 12, 64), ny=_log_int(rng, 12, 64),
                 steps=rng.randint(1, 10), persistent=rng.random() < 0.5)
    elif kind == "steps":  # 16 to 1023 a side
        c.update(nx=_log_int(rng, 16, 1023), ny=_log_int(rng, 16, 1001))
        c.update(steps=max(1, min(30, 4000000 // (c["nx"] * c["ny"]))),
                 tol=rng.choice(["fixed", "relative", "absolute"]))
    elif kind == "rollout":
        c.update(nx=_log_int(rng, 24, 192), ny=_log_int(rng, 24, 192), steps=rng.randint(4, 24), every=rng.randint(2, 8))
    elif kind in ("batch", "batch_rollout"):
        lo = _log_int(rng, 8, 48)
        c.update(lo=lo, hi=rng.randint(lo, 128 if kind == "batch" else 96), layout=rng.randint(1, 1000),
                 cloths=_log_int(rng, 8, 512 if kind == "batch" else 64))
        c.update(zip(("threads", "per_thread"), rng.choice([(1024, 1), (1024, 1), (512, 8)])))
        if kind == "batch":
            c.update(steps=rng.randint(10, 60))
        else:
            c.update(steps=rng.randint(3, 10), every=rng.randint(2, 5))
    else:
        c.update(nx=_log_int(rng, 16, 640), ny=_log_int(rng, 16, 640),
                 steps=1 if kind == "vgrid" else rng.choice([1, _log_int(rng, 1, 100)]) if kind == "verlet"
                 else rng.choice([1, rng.randint(1, 10)]))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=16)
def _grid(nx, ny, y0):
    """Rest positions of an nx x ny grid over the 4x4 square and its spring list."""
    from opencloth_amd import scenes

    X = scenes.grid_positions(nx, ny, 4.0, y0)
    return X, scenes.grid_springs(nx, ny, X, KS, KD)


@functools.lru_cache(maxsize=4)
def _layout(cloths, lo, hi, layout, diff):
    from opencloth_amd import scenes

    f = scenes.batch_diff_scene if diff else scenes.batch_scene
    return f(n_cloths=cloths, sides=(lo, hi), seed=layout)


def _noise(rng, n, width):
    return rng.standard_normal((n, 3), dtype=np.float32) * np.float32(width)


def _scene(case, seed):
    """(positions, velocities, springs, pins, StepParams, more) of a case."""
    import dataclasses

    from opencloth_amd import scenes

    rng = np.random.default_rng([int(seed), 17])
    kind = case["kind"]
    if kind in ("batch", "batch_rollout"):
        b = _layout(case["cloths"], case["lo"], case["hi"], case["layout"], kind == "batch_rollout")
        width = np.repeat(4.0 / (b.nx - 1), b.nx.astype(np.int64) * b.ny).astype(np.float32)[:, None]
        X = b.X + _noise(rng, len(b.X), 1e-3) * width
        V = _noise(rng, len(X), 1e-2)
        return X, V, b.springs, b.pinned, b.params, {"batch": b, "target": b.extra.get("target")}
    nx, ny = case["nx"], case["ny"]
    n = nx * ny
    if kind == "physics":
        # the demo's constants, the cloth already at the collider, so that the
        # contact and Provot passes have work from the first step
        base = scenes.demo_scene(21) if case["scene"] == "ie" else scenes.bw_demo_scene(21)
        X0 = scenes.grid_positions(nx, ny, 4.0, 2.6)
        sp = scenes.grid_springs(nx, ny, X0, (0.75, 0.75, 0.95), KD)
        X = X0 + _noise(rng, n, 1e-2 * 4.0 / (max(nx, ny) - 1))
        pins = np.zeros(n, np.uint8)
        pins[0] = pins[nx - 1] = 1
        p = dataclasses.replace(base.params, cg_persistent=bool(case["persistent"]))
        return X, _noise(rng, n, 1e-2), sp, pins, p, dict(base.extra)
    X0, sp = _grid(nx, ny, 0.0 if kind in ("steps", "rollout") else 2.6)
    X = X0 + _noise(rng, n, 1e-3 * 4.0 / (max(nx, ny) - 1))
    V = _noise(rng, n, 1e-2)
    pins = np.zeros(n, np.uint8)
    pins[:nx] = 1
    if kind == "steps":
        p = {"fixed": scenes.StepParams(dt=1.0 / 120.0, cg_max_iters=30, cg_tol=0.0, cg_tol_mode=scenes.TOL_NONE),
             "relative": scenes.StepParams(cg_max_iters=40, cg_tol=1e-4, cg_tol_mode=scenes.TOL_RELATIVE),
             "absolute": scenes.StepParams(cg_max_iters=10, cg_tol=1e-3, cg_tol_mode=scenes.TOL_ABSOLUTE)}[case["tol"]]
        return X, V, sp, pins, p, {}
    if kind == "rollout":
        p = scenes.StepParams(cg_max_iters=40, cg_tol=0.0, cg_tol_mode=scenes.TOL_NONE)
        ks = rng.uniform(30.0, 80.0, len(sp)).astype(np.float32)
        return X, V, sp, pins, p, {"ks": ks, "target": scenes.smooth_target(X0, 0)}
    if kind == "verlet":
        p = scenes.verlet_demo_scene(21)
        return X, (X - _noise(rng, n, 1e-4)).astype(np.float32), sp, pins, p.params, dict(p.extra)
    if kind == "vgrid":
        pins[:] = 0
        pins[0] = pins[nx - 1] = 1
        return X, (X - _noise(rng, n, 1e-4)).astype(np.float32), None, pins, scenes.vgrid_params(nx, ny), {}
    p = scenes.pbd_demo_scene(21)
    dist, bend = scenes.pbd_grid_constraints(nx, ny)
    mass = float(np.float32(1.0) / np.float32(n))
    return X, V, (dist, bend), pins, dataclasses.replace(p.params, mass=mass), dict(p.extra)


def prepare(case, seed):
    """The handle a program keeps, with its state in device memory."""
    from opencloth_amd import batch, cloth

    X, V, sp, pins, p, more = _scene(case, seed)
    kind = case["kind"]
    s = dict(case, X=X, V=V, more=more)
    if kind in ("batch", "batch_rollout"):
        b = more["batch"]
        s["h"] = batch.ClothBatch(b.nx, b.ny, X, sp, b.n_springs, pins, p, V)
        s["h"].set_schedule(case["threads"], case["per_thread"])
        s["ks"] = np.ascontiguousarray(sp["Ks"])
    elif kind in ("physics", "steps", "rollout"):
        s["h"] = cloth.ImplicitCloth(case["nx"], case["ny"], X, sp, pins, p, V)
    elif kind == "verlet":
        s["h"] = cloth.VerletCloth(case["nx"], case["ny"], X, sp, pins, p.mass, p.gravity, more["damping"], p.dt,
                                   p.ground_clamp, V)
    elif kind == "vgrid":
        import torch

        one = np.ones((len(X), 1), np.float32)
        s["h"] = cloth.VerletGrid(case["nx"], case["ny"], np.hstack([X, one]), np.hstack([V, one]), pins, p)
        s["vbo"] = torch.zeros(len(X), 4, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
    else:
        s["h"] = cloth.PBDCloth(X, sp[0], sp[1], pins, p, V)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    kind, h = s["kind"], s["h"]
    if kind == "physics":
        h.step_physics(s["steps"], s["more"]["ellipsoid"], s["more"]["provot_slack"])
    elif kind in ("steps", "batch"):
        h.step(s["steps"])
    elif kind in ("rollout", "batch_rollout"):
        h.set_spring_stiffness(s["more"]["ks"] if kind == "rollout" else s["ks"])
        h.set_state(s["X"], s["V"])
        h.rollout_forward(s["steps"], s["every"])
        X, V = h.get_state()
        g = h.rollout_backward(2.0 * (X - s["more"]["target"]))
        return {"x": X, "v": V, "ks": g[0], "x0": g[1], "v0": g[2]}
    elif kind == "vgrid":
        h.step(s["steps"], s["vbo"].data_ptr())
        h.synchronize()
        return {"vbo": s["vbo"]}
    else:
        h.step(s["steps"], s["more"]["ellipsoid"])
    X, V = h.get_state()
    return {"x": X, "v": V}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _sizes(case):
    """(vertices, springs) of a case."""
    if case["kind"] in ("batch", "batch_rollout"):
        from opencloth_amd import scenes

        u = scenes.uniform(case["layout"], 4 * case["cloths"]).reshape(4, case["cloths"])
        side = case["lo"] + np.floor(u[0] * (case["hi"] - case["lo"] + 1))
        return int((side ** 2).sum()), int((4 * side * (side - 1) + 2 * (side - 1) ** 2).sum())
    nx, ny = case["nx"], case["ny"]
    return nx * ny, 2 * (ny * (nx - 1) + nx * (ny - 1)) + 2 * (nx - 1) * (ny - 1)


def work(case):
    """State and constants read once, state (and gradients) written once;
    floating-point operations of every step.  A solve with a stopping test is
    counted with the 5 iterations that these cloths take on average."""
    N, S = _sizes(case)
    kind, steps = case["kind"], case["steps"]
    spring, pair = 60.0, 24.0  # one spring's force and Jacobian; one block times a vector, both ends
    its = {"fixed": 30.0, "rollout": 40.0, "batch_rollout": 12.0}.get(case.get("tol", kind), 5.0)
    solve = its * (pair * S + 30.0 * N)
    if kind in ("physics", "steps", "batch"):
        post = 12.0 * S if kind == "physics" else 0.0
        return {"bytes": 73.0 * N + 12.0 * S, "flops": steps * ((spring + pair) * S + post + solve + 30.0 * N)}
    if kind in ("rollout", "batch_rollout"):
        return {"bytes": 97.0 * N + 20.0 * S, "flops": steps * (3.0 * spring * S + 2.0 * solve + 60.0 * N)}
    if kind == "verlet":
        return {"bytes": 49.0 * N + 12.0 * S, "flops": steps * (35.0 * S + 30.0 * N)}
    if kind == "vgrid":
        return {"bytes": 65.0 * N, "flops": steps * (35.0 * S + 30.0 * N)}
    # two solver iterations of about 4 distance and 2 bending constraints per particle
    return {"bytes": 53.0 * N + 88.0 * N, "flops": steps * (2.0 * (4 * 35.0 + 2 * 50.0) * N + 120.0 * N)}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _f(v):
    """The float the library is given, as a double."""
    return float(np.float32(v))


class _Implicit64:
    """Implicit steps of one cloth or of many independent ones, in float64.
    Pair terms are C w = a w + b n (n.w), with n the spring's direction."""

    def __init__(self, springs, sizes, counts, pinned, p, dev, ks=None):
        import torch

        self.t, self.dev = torch, dev
        off = np.repeat(np.concatenate([[0], np.cumsum(sizes)[:-1]]), counts)
        self.p1 = torch.from_numpy(springs["p1"].astype(np.int64) + off).to(dev)
        self.p2 = torch.from_numpy(springs["p2"].astype(np.int64) + off).to(dev)
        self.L0, self.ks, self.kd = (torch.from_numpy(np.ascontiguousarray(v).astype(np.float64)).to(dev)
                                     for v in (springs["rest_length"], springs["Ks"] if ks is None else ks,
                                               springs["Kd"]))
        self.free = torch.from_numpy((pinned == 0).astype(np.float64)).to(dev)[:, None]
        self.sizes = torch.from_numpy(np.asarray(sizes, np.int64)).to(dev)
        self.cid = torch.repeat_interleave(torch.arange(len(sizes), device=dev), self.sizes)
        self.p, self.h, self.mass, self.c = p, _f(p.dt), _f(p.mass), _f(p.damping)
        self.md = self.mass - self.h * self.c
        self.g = torch.tensor([_f(v) for v in p.gravity], dtype=torch.float64, device=dev)
        self.dv = None

    def dot(self, a, b):
        return self.t.segment_reduce((a * b).sum(1), "sum", lengths=self.sizes)

    def gather(self, f):
        """Per-spring vectors added at the first end and subtracted at the second."""
        out = self.t.zeros(len(self.free), 3, dtype=self.t.float64, device=self.dev)
        return out.index_add_(0, self.p1, f).index_add_(0, self.p2, f, alpha=-1.0)

    def geometry(self, x):
        dp = x[self.p1] - x[self.p2]
        l = dp.norm(dim=1, keepdim=True)
        return dp / l, l[:, 0]

    def spring_force(self, x, v, ks):
        n, l = self.geometry(x)
        w = v[self.p1] - v[self.p2]
        return (-ks * (l - self.L0) + self.kd * (w * n).sum(1))[:, None] * n

    def stiffness(self, x, w, ks):
        """K w of every spring."""
        n, l = self.geometry(x)
        nw = (n * w).sum(1, keepdim=True) * n
        return ks[:, None] * (-w + (self.L0 / l)[:, None] * (w - nw))

    def matrix(self, x):
        n, l = self.geometry(x)
        h, lo = self.h, self.L0 / l
        self.n, self.a, self.b = n, (h * h * self.ks * (lo - 1.0))[:, None], (h * self.kd - h * h * self.ks * lo)[:, None]
        self.pinv = None
        if self.p.cg_jacobi:
            c = self.a + self.b * n * n
            dg = self.md - self.t.zeros_like(x).index_add_(0, self.p1, c).index_add_(0, self.p2, c)
            self.pinv = self.t.where(dg > 0, 1.0 / dg, self.t.ones_like(dg))

    def product(self, d):
        w = d[self.p1] - d[self.p2]
        return self.free * (self.md * d - self.gather(self.a * w + self.b * self.n * (self.n * w).sum(1, keepdim=True)))

    def solve(self, b, x):
        """Filtered conjugate gradients from x with the library's stopping tests, every cloth by its own."""
        t, p = self.t, self.p
        z_of = (lambda r: r) if self.pinv is None else (lambda r: self.pinv * r)
        r = self.free * (b - self.md * x) if x is None else self.free * b - self.product(x)
        d = z_of(r)
        delta = self.dot(r, d)
        limit = _f(p.cg_tol) ** 2 * (delta if p.cg_tol_mode == 1 else t.ones_like(delta))
        live = t.ones_like(delta, dtype=t.bool)
        for _ in range(p.cg_max_iters):
            if p.cg_tol_mode != 2:
                live = live & (delta > limit)
                if not bool(live.any()):
                    break
            q = self.product(d)
            sigma = self.dot(d, q)
            live = live & (sigma >= 0)
            alpha = t.where(live & (sigma > 0), delta / sigma, t.zeros_like(delta))[self.cid][:, None]
            x = x + alpha * d
            r = r - alpha * q
            z = z_of(r)
            new = self.dot(r, z)
            beta = t.where(live & (delta > 0), new / delta, t.zeros_like(delta))[self.cid][:, None]
            d = t.where(live[self.cid][:, None], z + beta * d, d)
            delta = t.where(live, new, delta)
        return x

    def step(self, x, v):
        h = self.h
        f = self.free * (self.mass * self.g + self.c * v) + self.gather(self.spring_force(x, v, self.ks))
        f = f + h * self.gather(self.stiffness(x, v[self.p1] - v[self.p2], self.ks))
        self.matrix(x)
        self.dv = self.solve(h * f, self.t.zeros_like(x) if self.dv is None else self.dv)
        v = v + self.dv
        x = x + h * v
        if self.p.ground_clamp:
            x[:, 1].clamp_(min=0.0)
        return x, v

    def adjoint(self, x, v, dv, gx, gv, gks):
        """Gradients before the step (x, v) -> (x + h(v + dv), v + dv)."""
        t, h = self.t, self.h
        gvt = gv + h * gx
        self.matrix(x)
        mu = self.solve(gvt, t.zeros_like(x))
        x, v, ks = (q.detach().clone().requires_grad_(True) for q in (x, v, self.ks))
        with t.enable_grad():
            n, _ = self.geometry(x)
            u, wp = mu[self.p1] - mu[self.p2], dv[self.p1] - dv[self.p2]
            w = v[self.p1] - v[self.p2] + wp
            J = (h * (u * self.spring_force(x, v, ks)).sum() + h * h * (u * self.stiffness(x, w, ks)).sum()
                 + h * (self.kd * (u * n).sum(1) * (n * wp).sum(1)).sum() + h * self.c * (self.free * mu * v).sum())
        jx, jv, jk = t.autograd.grad(J, (x, v, ks))
        return gx + jx, gvt + jv, gks + jk


def _collide64(t, x, w, e, to_surface):
    """The ellipsoid pass: points inside are pushed out; w becomes zero, or the
    new position, there."""
    Mi, M = (t.from_numpy(e[k].astype(np.float64)).to(x.device).reshape(4, 4) for k in ("Minv", "M"))
    d = x @ Mi[:3, :3] + Mi[3, :3] - t.from_numpy(e["center"].astype(np.float64)).to(x.device)
    dist = d.norm(dim=1, keepdim=True)
    inside = dist < 1.0
    d = (e["radius"] - dist) * d / dist
    rows = M[:3, :3].T
    y = x + d @ (rows / (rows * rows).sum(1, keepdim=True)).T
    x = t.where(inside, y, x)
    return x, t.where(inside, x if to_surface else t.zeros_like(w), w)


def _colours(n, cons, arity):
    """Constraint ids by colour: each takes the lowest colour not yet used at its particles, in list order."""
    used, col = [0] * n, []
    for ps in zip(*(cons["p%d" % (k + 1)].tolist() for k in range(arity))):
        m = 0
        for a in ps:
            m |= used[a]
        bit = ~m & (m + 1)
        for a in ps:
            used[a] |= bit
        col.append(bit.bit_length() - 1)
    col = np.asarray(col)
    return [np.flatnonzero(col == k) for k in range(int(col.max()) + 1)]


def _pbd64(case, X, V, cons, pins, p, more, t, dev):
    up = lambda a: t.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    x, v = up(X.astype(np.float64)), up(V.astype(np.float64))
    mass, dt, n = _f(p.mass), _f(p.dt), len(X)
    w = up(np.where(pins != 0, 0.0, 1.0 / mass))[:, None]
    gd = min(_f(p.global_damping), 1.0)
    kp = lambda k: min(1.0, 1.0 - (1.0 - _f(k)) ** (1.0 / p.solver_iterations))  # noqa: E731
    third = _f(0.3333)
    fam = []
    for c, arity in zip(cons, (2, 3)):
        for ids in _colours(n, c, arity):
            q = [up(c["p%d" % (k + 1)][ids].astype(np.int64)) for k in range(arity)]
            if arity == 2:
                rest = (x0 := up(X.astype(np.float64)))[q[0]].sub(x0[q[1]]).norm(dim=1, keepdim=True)
            else:
                x0 = up(X.astype(np.float64))
                rest = (x0[q[2]] - third * (x0[q[0]] + x0[q[1]] + x0[q[2]])).norm(dim=1, keepdim=True)
            fam.append((q, rest, kp(c["k"][0])))
    for _ in range(case["steps"]):
        f = (w > 0) * t.tensor([_f(g) for g in p.gravity], dtype=t.float64, device=dev)
        v = v * gd + f * dt * w
        xc, vc = x.mean(0), v.mean(0)
        R = x - xc
        L = t.linalg.cross(R, mass * v).sum(0)
        eye = t.eye(3, dtype=t.float64, device=dev)
        inertia = eye + mass * ((R * R).sum() * eye - R.T @ R)
        om = t.linalg.solve(inertia, L)
        v = v + _f(p.k_damp) * (vc + t.linalg.cross(om.expand_as(R), R) - v)
        y = t.where(w > 0, x + v * dt, x)
        for _ in range(p.solver_iterations):
            for q, rest, k in fam:
                if len(q) == 2:
                    a, b = q
                    d = y[a] - y[b]
                    l = d.norm(dim=1, keepdim=True)
                    im = w[a] + w[b]
                    go = (l > 1e-7) & (im > 1e-7)
                    dP = t.where(go, (l - rest) / im * (d / l) * k, t.zeros_like(d))
                    y[a], y[b] = y[a] - dP * w[a], y[b] + dP * w[b]
                else:
                    a, b, c = q
                    d = y[c] - third * (y[a] + y[b] + y[c])
                    f = d * (1.0 - (_f(gd * 0.01) + rest) / d.norm(dim=1, keepdim=True))
                    ws = (w[a] + w[b] + 2.0 * w[c]).clamp(min=1e-300)  # 0 where all three are pinned
                    y[a], y[b], y[c] = (y[a] + k * 2 * w[a] / ws * f, y[b] + k * 2 * w[b] / ws * f,
                                        y[c] - k * 4 * w[c] / ws * f)
            if p.ground:
                y[:, 1].clamp_(min=0.0)
        y, v = _collide64(t, y, v, more["ellipsoid"], False)
        v = (y - x) / dt
        x = y
    return {"x": x.cpu().numpy(), "v": v.cpu().numpy()}


def _vgrid64(case, X, XL, pins, p, t, dev):
    nx, ny, dt, mass = case["nx"], case["ny"], _f(p["dt"]), _f(p["mass"])
    up = lambda a: t.from_numpy(a.astype(np.float64)).to(dev).reshape(ny, nx, -1)  # noqa: E731
    x, xl, free = up(X), up(XL), up((pins == 0)[:, None])
    stencil = [(1, 0), (0, -1), (-1, 0), (0, 1), (1, -1), (-1, -1), (-1, 1), (1, 1), (2, 0), (0, -2), (-2, 0), (0, 2)]
    for _ in range(case["steps"]):
        v = (x - xl) / dt
        F = t.tensor([_f(g) for g in p["gravity"]], dtype=t.float64, device=dev) * mass + v * _f(p["damping"])
        for k, (dx, dy) in enumerate(stencil):
            at = (slice(max(0, -dy), ny - max(0, dy)), slice(max(0, -dx), nx - max(0, dx)))
            to = (slice(max(0, dy), ny - max(0, -dy)), slice(max(0, dx), nx - max(0, -dx)))
            d, dv = x[at] - x[to], v[at] - v[to]
            l = d.norm(dim=2, keepdim=True)
            rest = math.hypot(dx * _f(p["spacing"][0]), dy * _f(p["spacing"][1]))
            F[at] += (-_f(p["ks"][k // 4]) * (l - rest) + _f(p["kd"][k // 4]) * (dv * d).sum(2, keepdim=True) / l) * d / l
        xc = x.clone()
        xc[..., 1].clamp_(min=0.0)
        x, xl = 2.0 * xc - xl + free * F / mass * dt * dt, xc
    return {"vbo": np.concatenate([x.reshape(-1, 3).cpu().numpy(), np.ones((nx * ny, 1))], 1)}


def exact(case, seed):
    import torch as t

    dev = "cuda" if t.cuda.is_available() else "cpu"
    X, V, sp, pins, p, more = _scene(case, seed)
    kind = case["kind"]
    with t.no_grad():
        if kind == "pbd":
            return _pbd64(case, X, V, sp, pins, p, more, t, dev)
        if kind == "vgrid":
            return _vgrid64(case, X, V, pins, p, t, dev)
        b = more.get("batch")
        sizes, counts = (b.nx.astype(np.int64) * b.ny, b.n_springs) if b is not None else ([len(X)], [len(sp)])
        s = _Implicit64(sp, sizes, counts, pins, p, dev, more.get("ks"))
        x, v = (t.from_numpy(q.astype(np.float64)).to(dev) for q in (X, V))
        if kind == "verlet":
            xl, damp, dt = v, _f(more["damping"]), _f(p.dt)
            for _ in range(case["steps"]):
                vel = (x - xl) / dt
                F = s.free * (s.mass * s.g + s.gather(s.spring_force(x, vel, s.ks))) + damp * vel
                x, xl = x + (x - xl) + dt * dt / s.mass * F, x
                x[:, 1].clamp_(min=0.0)
                x, xl = _collide64(t, x, xl, more["ellipsoid"], True)
            return {"x": x.cpu().numpy(), "v": xl.cpu().numpy()}
        trace = []
        for _ in range(case["steps"]):
            x1, v1 = s.step(x, v)
            if kind in ("rollout", "batch_rollout"):
                trace.append((x, v, s.dv))
            x, v = x1, v1
            if kind == "physics":
                x, v = _collide64(t, x, v, more["ellipsoid"], False)
                n, l = s.geometry(x)
                over = l - s.L0 * _f(more["provot_slack"])
                dP = t.where(over > 0, over / 2, t.zeros_like(over))[:, None] * n
                f1, f2 = s.free[s.p1], s.free[s.p2]
                v = v.index_add(0, s.p1, -dP * f1).index_add(0, s.p2, dP * t.maximum(1.0 - f1, f2))
        out = {"x": x.cpu().numpy(), "v": v.cpu().numpy()}
        if trace:
            gx = 2.0 * (x - t.from_numpy(more["target"].astype(np.float64)).to(dev))
            gv, gks = t.zeros_like(gx), t.zeros_like(s.ks)
            while trace:
                gx, gv, gks = s.adjoint(*trace.pop(), gx, gv, gks)
            out.update(ks=gks.cpu().numpy(), x0=gx.cpu().numpy(), v0=gv.cpu().numpy())
        return out
