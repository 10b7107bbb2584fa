"""The work that programs have this library do, as cases that can be timed.

A case is a dict of plain values; `kind` names the calling pattern:

  frame    an interactive program's loop (the reference's, scene.cpp:267-276):
           one simulate(), then the vertex buffer of that frame
  rollout  an offline program: a run of steps, then the state is read
  batch    many independent instances stepped together, then every state read
  adjoint  one gradient of a rollout: forward, then backward
  query    points tested against a body (host arrays in and out)
  posed    a program that animates the body itself: new body vertices, one
           simulate(), then the vertex buffer

Cloths are square grids of `side` vertices a side with the repository's
structural, shear and bend springs ("grid"), or the same sheet as a triangle
mesh with mesh springs and the reference's constants ("mesh").  Bodies are the
icosphere ("sphere", `detail` = subdivision level) or the twelve-capsule union
("capsules", `detail` = segments around), static, refitted or rebuilt every
frame.  Sheets are held along their edges, so that they stay on the body
however long a program runs; `settle` steps are run before the first pass, so
that the passes see the cloth in contact (0: the sheet starts to fall).
"""
import numpy as np
import torch

from simulator_amd import _lib as L
from simulator_amd import batch as B
from simulator_amd import scene as S
from simulator_amd.adjoint import Adjoint
from simulator_amd.simulator import Simulator

MODES = {"static": L.CC_BODY_STATIC, "refit": L.CC_BODY_REFIT, "rebuild": L.CC_BODY_REBUILD}


def listed():
    def case(name, kind, **more):
        return dict(name=name, kind=kind, **more)

    return [
        # the smallest call: one frame of the 64x64 cloth on a static sphere; launches and latency
        case("frame_small", "frame", cloth="grid", side=64, body="sphere", detail=4, mode="static", settle=400),
        # a garment-sized OBJ-like mesh (about 17k vertices, irregular spring counts) on a static body
        case("frame_mesh", "frame", cloth="mesh", side=130, body="sphere", detail=5, mode="static", settle=480),
        # the garment workload, interactive: 111x111 over 50,688 triangles rebuilt every frame
        case("frame_garment", "frame", cloth="grid", side=111, body="capsules", detail=64, mode="rebuild", settle=400),
        # the headline workload, interactive: 512x512 over 501,120 triangles refitted every frame
        case("frame_large", "frame", cloth="grid", side=512, body="capsules", detail=144, mode="refit", settle=600),
        # the same three workloads as offline runs: whole blocks of steps, then the state is read
        case("rollout_small", "rollout", cloth="grid", side=64, body="sphere", detail=4, mode="static", settle=400,
             steps=200),
        case("rollout_garment", "rollout", cloth="grid", side=111, body="capsules", detail=64, mode="rebuild",
             settle=400, steps=100),
        case("rollout_large", "rollout", cloth="grid", side=512, body="capsules", detail=144, mode="refit",
             settle=600, steps=200),
        # the batched workload: 256 uneven instances, every body rebuilt every frame
        case("batch_256", "batch", count=256, mode="rebuild", settle=320, steps=128),
        # a few instances with refitted bodies, a run that is no whole number of graph blocks
        case("batch_16", "batch", count=16, mode="refit", settle=320, steps=50),
        # the differentiable workload: 128x128, 200 steps, checkpoints every 20
        case("adjoint_128", "adjoint", side=128, steps=200, ckpt=20),
        # a caller's own points against a body of the garment workload's size
        case("query_20000", "query", points=20000, body="capsules", detail=64),
        # a body animated by the caller: new vertices every frame
        case("posed_garment", "posed", cloth="grid", side=111, body="capsules", detail=64, mode="static",
             settle=400),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    def scene(most):
        kind = rng.choice(["grid", "grid", "mesh"])
        body, mode = rng.choice([("sphere", "static"), ("capsules", "static"), ("capsules", "refit"),
                                 ("capsules", "rebuild")])
        detail = rng.randint(3, 6) if body == "sphere" else 4 * log(4, 36 if mode == "refit" else 20)
        side = log(24, most) if kind == "grid" else log(24, min(most, 240))
        return dict(cloth=kind, side=side, body=body, detail=detail, mode=mode, settle=rng.choice([0, 400, 500, 600]))

    kind = rng.choice(["frame", "frame", "rollout", "rollout", "batch", "adjoint", "query", "posed"])
    if kind == "frame":
        return dict(kind=kind, **scene(512))
    if kind == "rollout":
        return dict(kind=kind, **scene(360), steps=log(24, 200))
    if kind == "batch":
        return dict(kind=kind, count=log(2, 64), mode=rng.choice(["static", "refit", "rebuild", "rebuild"]),
                    settle=rng.choice([0, 320]), steps=log(8, 100))
    if kind == "adjoint":
        return dict(kind=kind, side=log(24, 160), steps=log(20, 200), ckpt=rng.randint(5, 40))
    if kind == "query":
        body = rng.choice(["sphere", "capsules"])
        return dict(kind=kind, points=log(500, 60000), body=body,
                    detail=rng.randint(3, 6) if body == "sphere" else 4 * log(4, 30))
    return dict(kind=kind, cloth="grid", side=log(24, 200), body="capsules", detail=4 * log(4, 20), mode="static",
                settle=400)


# ------------------------------------------------------------------ inputs


def _edges(side):
    j = np.arange(side)
    return np.unique(np.concatenate([j, j + side * (side - 1), j * side, j * side + side - 1])).astype(np.uint32)


def _body(case, seed):
    mode = MODES[case.get("mode", "static")]
    if case["body"] == "sphere":
        return S.sphere_body(case["detail"])
    d = case["detail"]
    # the repository's tessellations (64, 14, 6) and (144, 64, 18) at their own sizes
    nring, ncyl = {64: (14, 6), 144: (64, 18)}.get(d, (max(2, d // 4), max(2, d // 8)))
    return S.capsules(d, nring, ncyl, mode, seed=7 + seed % 1000)


def _scene(case, seed):
    side, body = case["side"], _body(case, seed)
    y0 = 1.0 if case["settle"] else 1.25      # above every body: no contact in the first passes
    if case["cloth"] == "mesh":
        pos = S.grid_cloth(side, side, 1.0 / (side - 1), 0.83 if case["settle"] else y0, 1e-4, seed)
        sc = S.mesh_scene("mesh", pos, S.grid_faces(side, side), body.verts, body.tris, body.normals)
        sc.body = body
    else:
        big = case["mode"] == "refit" and side >= 300
        sc = S.grid_scene("grid", side, 5e-4 if big else 1e-3, 0, body, seed=seed, y0=y0,
                          box_depth=0.01 if case["body"] == "sphere" else 0.002)
        sc.faces = S.grid_faces(side, side)
    sc.pins = _edges(side)
    return sc


def _poses(body, seed):
    """Poses of the body as its owner animates it: a sway about the y axis."""
    rng = np.random.default_rng(seed)
    out = []
    for k in range(4):
        a = 0.05 * np.sin(1.5 * k + rng.uniform(0, 6.28))
        c, s = np.cos(a), np.sin(a)
        R = np.array([[c, 0, s], [0, 1, 0], [-s, 0, c]])
        P = np.array([0.5, 0.6, 0.0])
        out.append(np.ascontiguousarray((body.verts - P) @ R.T + P, np.float32))
    return out


def _sizes(count):
    """(cloth side, capsule segments) of the batch's instances: the sides and
    tessellations that the repository's batched workload draws."""
    rng = np.random.default_rng(0)
    lo, hi = np.log(B.SIDE_RANGE[0]), np.log(B.SIDE_RANGE[1])
    return [(int(round(float(np.exp(rng.uniform(lo, hi))))),
             4 * int(rng.integers(B.CAPSULE_S[0] // 4, B.CAPSULE_S[1] // 4 + 1))) for _ in range(count)]


def _batch_scenes(case, seed):
    """The batched workload's instances (simulator_amd.batch.instances), their
    sizes the same for every seed."""
    rng = np.random.default_rng(seed)
    scs = []
    for k, (side, s) in enumerate(_sizes(case["count"])):
        ks = tuple(float(b * rng.uniform(0.7, 1.3)) for b in B.K_BASE)
        bseed = int(rng.integers(1, 2**31 - 1))
        v, t, nrm, caps = S.capsule_body(B.BATCH_CAPS, 0.04, 0.15, *S.CAPSULE_BOX, s, s // 4, s // 4, bseed)
        body = S.Body(v, t, nrm, MODES[case["mode"]], True, caps, S._motion(bseed))
        sc = S.grid_scene("batched", side, 1e-3, 0, body, k=ks, box_depth=0.002, seed=seed + k,
                          y0=1.0 if case["settle"] else 1.25)
        sc.pins = _edges(side)
        scs.append(sc)
    return scs


def _adjoint_inputs(case, seed):
    """The sheet tossed up a little over the sphere (it does not reach it
    within 200 steps), the loss weights, and the parameters under study."""
    rng = np.random.default_rng(seed)
    n = case["side"] ** 2
    v0 = (np.array([rng.uniform(-0.1, 0.1), rng.uniform(0.1, 0.2), rng.uniform(-0.1, 0.1)])
          + rng.normal(scale=1e-3, size=(n, 3))).astype(np.float32)
    g = rng.normal(size=(n, 3)).astype(np.float32)
    theta = np.array([1000.0, 500.0, 100.0, -0.02, 1.0]) * np.append(rng.uniform(0.8, 1.2, 4), 1.0)
    return v0, g, theta


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("frame", "rollout", "posed"):
        sc = _scene(case, seed)
        sim = Simulator.from_scene(sc)
        st = {"case": case, "sim": sim}
        if kind != "rollout":
            sim.set_faces(sc.faces)
            st["vbo"] = torch.zeros(7 * sc.n, dtype=torch.float32, device="cuda")
        if kind == "posed":
            st["poses"], st["k"] = _poses(sc.body, seed), 0
        torch.cuda.synchronize()
        sim.simulate(case["settle"])
        sim.synchronize()
        return st
    if kind == "batch":
        scs = _batch_scenes(case, seed)
        b = B.Batch(scs)
        n = sum(sc.n for sc in scs)
        b.simulate(case["settle"])
        b.synchronize()
        return {"case": case, "batch": b, "out": [np.zeros((n, 3), np.float32) for _ in range(3)]}
    if kind == "adjoint":
        sc = S.grid_scene("adjoint", case["side"], 1e-3, case["steps"], S.sphere_body(), seed=seed)
        sim = Simulator.from_scene(sc)
        v0, g, theta = _adjoint_inputs(case, seed)
        return {"case": case, "adj": Adjoint(sim, case["steps"], case["ckpt"]), "x0": sc.pos, "v0": v0, "g": g,
                "theta": theta}
    body = _body(case, seed)
    rng = np.random.default_rng(seed)
    one = (np.zeros(2, np.uint32), np.zeros(0, L.SPRING_DTYPE))
    sim = Simulator(np.zeros((1, 3), np.float32), [one], body, S.params(box_depth=0.005))
    # points about the surface, as the vertices of a garment on the body are
    v = body.verts[rng.integers(0, body.verts.shape[0], case["points"])]
    pts = (v + rng.normal(scale=3e-3, size=v.shape)).astype(np.float32)
    return {"case": case, "sim": sim, "pts": pts}


# -------------------------------------------------------------------- runs


def run(state):
    kind = state["case"]["kind"]
    if kind in ("frame", "posed"):
        sim, vbo = state["sim"], state["vbo"]
        if kind == "posed":
            state["k"] = (state["k"] + 1) % len(state["poses"])
            sim.set_body_vertices(state["poses"][state["k"]])
        sim.simulate(1)
        sim.cuda_update_vbo(vbo.data_ptr(), 4 * vbo.numel())
        return vbo
    if kind == "rollout":
        state["sim"].simulate(state["case"]["steps"])
        return state["sim"].get_state()
    if kind == "batch":
        b, out = state["batch"], state["out"]
        b.simulate(state["case"]["steps"])
        o = 0
        for k, n in enumerate(b.sizes):
            for whole, part in zip(out, b.get_state(k)):
                whole[o:o + n] = part
            o += n
        return out
    if kind == "adjoint":
        adj = state["adj"]
        xf = adj.forward(state["x0"], state["v0"], state["theta"])
        dth, dv0, dx0 = adj.backward(state["g"])
        return {"x": xf, "dtheta": dth, "dv0": dv0, "dx0": dx0}
    return state["sim"].collide_points(state["pts"])


# -------------------------------------------------------------------- work
# Payload bytes: 12 B per vector, 4 B per index or scalar, 8 B per spring
# record, each input read once and each output written once.


def _springs(case_cloth, side):
    if case_cloth == "mesh":      # edges and opposite corners of two triangles a cell, both directions
        e = 2 * side * (side - 1) + (side - 1) ** 2
        return 2 * e + 2 * (e - 4 * (side - 1))
    return 2 * (2 * side * (side - 1) + 2 * (side - 1) ** 2 + 2 * side * (side - 2))


def _body_size(case):
    if case["body"] == "sphere":
        return 10 * 4 ** case["detail"] + 2, 20 * 4 ** case["detail"]
    d = case["detail"]
    nring, ncyl = {64: (14, 6), 144: (64, 18)}.get(d, (max(2, d // 4), max(2, d // 8)))
    rows = 2 * nring + ncyl - 1
    return 12 * (d * rows + 2), 12 * 2 * d * rows


def _update_bytes(mode, nv, m):
    return {"static": 0, "refit": 72 * m + 36 * nv, "rebuild": 156 * m + 36 * nv}[mode]


def _step_work(n, springs, mode, nv, m):
    return 72 * n + 12 * n + 8 * springs + _update_bytes(mode, nv, m), 45 * springs + 120 * n + 60 * m * (mode != "static")


def work(case):
    kind = case["kind"]
    if kind in ("frame", "rollout", "posed"):
        side = case["side"]
        n, (nv, m) = side * side, _body_size(case)
        by, fl = _step_work(n, _springs(case["cloth"], side), case["mode"], nv, m)
        if kind == "rollout":
            return {"bytes": by * case["steps"] + 36 * n, "flops": fl * case["steps"]}
        faces = 2 * (side - 1) ** 2
        by, fl = by + 28 * n + 24 * faces, fl + 40 * faces + 30 * n
        if kind == "posed":
            by, fl = by + 156 * m + 12 * nv, fl + 100 * m
        return {"bytes": by, "flops": fl}
    if kind == "batch":
        by = fl = 0
        for side, s in _sizes(case["count"]):
            m = B.capsule_triangles(s)
            b, f = _step_work(side ** 2, _springs("grid", side), case["mode"], m // 2 + 2 * B.BATCH_CAPS, m)
            by, fl = by + b * case["steps"] + 36 * side ** 2, fl + f * case["steps"]
        return {"bytes": by, "flops": fl}
    if kind == "adjoint":
        n, e = case["side"] ** 2, _springs("grid", case["side"])
        by, fl = _step_work(n, e, "static", 0, 0)
        # a step forward; a step back reads the state, the normals and the adjoint and writes the adjoint
        return {"bytes": (by + 96 * n + 8 * e) * case["steps"] + 84 * n, "flops": (fl + 160 * e + 60 * n) * case["steps"]}
    nv, m = _body_size(case)
    return {"bytes": 41 * case["points"] + 52 * m, "flops": 200 * case["points"]}


# ------------------------------------------------------------------- exact
# The same steps in 64 bits with torch, for the cases that do not reach the
# body: the constants are the 32-bit ones that the library is given.


class _Exact:
    def __init__(self, sc, theta=None):
        p, dev = sc.params, "cuda" if torch.cuda.is_available() else "cpu"
        self.dt, self.mass, self.kd, self.eps = p.dt, p.mass, p.kd, p.eps
        self.g = torch.tensor(list(p.gravity), dtype=torch.float64, device=dev) * p.mass
        self.theta = torch.tensor([p.k[0], p.k[1], p.k[2], p.damp, p.rest_scale] if theta is None else
                                  [float(np.float32(t)) for t in theta], dtype=torch.float64, device=dev)
        src, dst, rest, kind = [], [], [], []
        for t, (row, col) in enumerate(sc.springs):
            src.append(np.repeat(np.arange(sc.n), np.diff(row.astype(np.int64))))
            dst.append(col["end"].astype(np.int64))
            rest.append(col["original"].astype(np.float64))
            kind.append(np.full(col.shape[0], t))
        to = lambda a, dt: torch.from_numpy(np.concatenate(a)).to(dev, dt)  # noqa: E731
        self.src, self.dst, self.kind = to(src, torch.int64), to(dst, torch.int64), to(kind, torch.int64)
        self.rest = to(rest, torch.float64)
        self.free = torch.ones(sc.n, 1, dtype=torch.float64, device=dev)
        self.free[torch.from_numpy(np.asarray(sc.pins, np.int64)).to(dev)] = 0

    def step(self, p, q):
        v = (p - q) / self.dt
        d = p[self.src] - p[self.dst] + self.eps
        dv = v[self.src] - v[self.dst]
        ln = d.norm(dim=1, keepdim=True)
        alpha = (-self.theta[self.kind] * (ln[:, 0] - self.rest * self.theta[4]))[:, None] \
            + self.kd * (dv * d).sum(1, keepdim=True) / ln
        f = torch.zeros_like(p).index_add(0, self.src, alpha * d / ln) + self.g + self.theta[3] * v
        return p + self.free * (p - q + f * (self.dt ** 2 / self.mass)), p


def _falls(steps, dt):
    return 0.5 * 9.8 * (steps * dt) ** 2 * 1.05


def exact(case, seed):
    kind = case["kind"]
    host = lambda t: t.detach().cpu().numpy()  # noqa: E731
    if kind == "adjoint":
        if case["side"] ** 2 * case["steps"] > 128 * 128 * 200:
            return None
        sc = S.grid_scene("adjoint", case["side"], 1e-3, case["steps"], S.sphere_body(), seed=seed)
        v0, g, theta = _adjoint_inputs(case, seed)
        E = _Exact(sc, theta)
        dev = E.g.device
        E.theta.requires_grad_()
        v = torch.from_numpy(v0).to(dev, torch.float64).requires_grad_()
        x = torch.from_numpy(np.ascontiguousarray(sc.pos)).to(dev, torch.float64).requires_grad_()
        p, q = x, x - v * E.dt
        for _ in range(case["steps"]):
            p, q = E.step(p, q)
        dth, dv, dx = torch.autograd.grad((p * torch.from_numpy(g).to(dev, torch.float64)).sum(), [E.theta, v, x])
        return {"x": host(p), "dtheta": host(dth), "dv0": host(dv), "dx0": host(dx)}
    if kind not in ("frame", "rollout", "batch") or case["settle"]:
        return None
    steps = case.get("steps", 1)
    scs = _batch_scenes(case, seed) if kind == "batch" else [_scene(case, seed)]
    if _falls(steps, scs[0].params.dt) > 0.04 or case.get("count", 1) > 32:
        return None
    outs = []
    for sc in scs:
        E = _Exact(sc)
        p = torch.from_numpy(np.ascontiguousarray(sc.pos)).to(E.g.device, torch.float64)
        q = p
        for _ in range(steps):
            p, q = E.step(p, q)
        outs.append((p, q))
    x, xp = (torch.cat([o[k] for o in outs]) for k in (0, 1))
    if kind != "frame":
        return (host(x), host(xp), np.zeros(x.shape)) if kind == "rollout" else [host(x), host(xp), np.zeros(x.shape)]
    # the vertex buffer: positions with w = 1, then the sums of the adjacent unit face normals, normalised
    f = torch.from_numpy(scs[0].faces.astype(np.int64)).to(x.device)
    a, b, c = x[f[:, 0]], x[f[:, 1]], x[f[:, 2]]
    fn = torch.nn.functional.normalize(torch.linalg.cross(b - a, c - a), dim=1)
    n = torch.zeros_like(x)
    for k in range(3):
        n = n.index_add(0, f[:, k], fn)
    n = torch.nn.functional.normalize(n, dim=1)
    return torch.cat([torch.cat([x, torch.ones_like(x[:, :1])], 1).reshape(-1), n.reshape(-1)])
