"""Performance cases of the batched planners, link(), nearest neighbours and
the collision surrogate, through the entry points of ``mpt_amd.Context``.

Every case runs with the launch shapes a context starts with.  Planner cases
are whole solves from the start state to a tree size, which is what a
planning program does; the batched downcalls (link, kNN) take device buffers,
as a program that drives its own loop does, except for the small host-array
call.  Sizes are those of the benchmark, the tests and the demo scenes.
"""
from __future__ import annotations

import dataclasses
import functools
import math

import numpy as np
import torch

import mpt_amd
from mpt_amd import scenes, surrogate

INF = math.inf
ORDERS = {"reference": mpt_amd.ORDER_REFERENCE, "surrogate": mpt_amd.ORDER_SURROGATE}
METRICS = {"l1": mpt_amd.METRIC_L1, "l2": mpt_amd.METRIC_L2, "se3": mpt_amd.METRIC_SE3}
# FLOPs of one joint of a planar arm's forward kinematics, and mean waypoint
# checks of one planner edge of the arm (counted on the benchmark's batch)
FK_FLOPS, ARM_CHECKS = 50, 82
# layers of the surrogate: 64-128-128-128-1
MLP = ((64, 128), (128, 128), (128, 128), (128, 1))
MLP_MACS = sum(i * o for i, o in MLP)


def listed():
    return [
        # a first plan in a small 2-D scene: a few short iterations, where
        # launches and read-backs count
        {"name": "prrt_boxes_b256", "kind": "prrt", "scene": "boxes", "batch": 256, "nodes": 2000,
         "order": "reference"},
        # exploring a large occupancy map with the batch the planner is meant for
        {"name": "prrt_grid4096_b8192", "kind": "prrt", "scene": "grid", "size": 4096, "batch": 8192, "nodes": 20000,
         "order": "reference"},
        # the benchmark's planner: a 20-link arm, surrogate-ordered checks
        {"name": "prrt_arm20_b8192", "kind": "prrt", "scene": "arm", "links": 20, "disks": 200, "batch": 8192,
         "nodes": 10000, "order": "surrogate"},
        # asymptotically optimal planning in 2-D with the default k-nearest formula
        {"name": "star_boxes_b1024", "kind": "star", "scene": "boxes", "batch": 1024, "nodes": 5000, "k": 0,
         "radius_lists": False},
        # optimal planning of a rigid body among 50 000 triangles, k = 20
        {"name": "star_se3_b4096", "kind": "star", "scene": "mesh", "robot": 500, "env": 50000, "batch": 4096,
         "nodes": 5000, "k": 20, "radius_lists": False},
        # the edges of one path, checked from host arrays (shortcutting, replay)
        {"name": "link_arm20_host_64", "kind": "link", "scene": "arm", "links": 20, "disks": 200, "n": 64,
         "order": "reference", "host": True},
        # one planner batch of arm edges decided for a caller's own loop
        {"name": "link_arm20_8192", "kind": "link", "scene": "arm", "links": 20, "disks": 200, "n": 8192,
         "order": "reference", "host": False},
        # roadmap-sized edge validation on an occupancy grid
        {"name": "link_grid4096_2p20", "kind": "link", "scene": "grid", "size": 4096, "n": 1 << 20,
         "order": "reference", "host": False},
        # one batch of rigid-body edges among triangles
        {"name": "link_se3_4096", "kind": "link", "scene": "mesh", "robot": 500, "env": 50000, "n": 4096,
         "order": "reference", "host": False},
        # nearest tree node of a batch of arm samples on a grown tree
        {"name": "knn_l1_20d_1e5", "kind": "knn", "metric": "l1", "dim": 20, "nodes": 100000, "queries": 8192, "k": 1},
        # neighbour lists for a dense roadmap
        {"name": "knn_l2_7d_1e6_k20", "kind": "knn", "metric": "l2", "dim": 7, "nodes": 1000000, "queries": 65536,
         "k": 20},
        # fitting the surrogate to labelled waypoints, in the batches it is trained with
        {"name": "surrogate_train_2p15", "kind": "train", "rows": 1 << 15, "batch": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges."""
    kind = rng.choice(["prrt", "prrt", "star", "link", "link", "knn", "knn", "train"])
    if kind == "train":
        batch = rng.choice([256, 512, 1024])
        return {"kind": kind, "rows": batch * rng.randint(2, (1 << 15) // batch), "batch": batch}
    if kind == "knn":
        metric = rng.choice(["l1", "l2", "l2", "se3"])
        queries = _log(rng, 256, 65536)
        if metric == "l1":
            dim, k, most = rng.choice([8, 10, 12, 16, 20]), 1, 1e9
        elif metric == "l2":
            dim, k, most = rng.randint(2, 8), rng.choice([1, 1, 10, 20]), 6e10 if queries > 4096 else 4e9
        else:
            dim, k, most = 7, rng.choice([1, 20]), 1e8
        return {"kind": kind, "metric": metric, "dim": dim, "nodes": _log(rng, 1000, min(1e6, most / queries)),
                "queries": queries, "k": k}
    if kind == "star":
        if rng.random() < 0.3:
            batch = _log(rng, 512, 4096)
            return {"kind": kind, "scene": "mesh", "robot": rng.choice([120, 250, 500]),
                    "env": rng.choice([6000, 20000, 50000]), "batch": batch, "nodes": min(5000, batch + rng.randint(0, batch)),
                    "k": rng.choice([10, 20]), "radius_lists": False}
        batch = _log(rng, 128, 1024)
        c = {"kind": kind, "scene": "boxes", "batch": batch, "nodes": batch * rng.randint(2, 5)}
        lists = rng.random() < 0.3
        return {**c, "k": 0 if lists else rng.choice([0, 10, 20]), "radius_lists": lists}
    scene = rng.choice(["boxes", "grid", "arm", "arm"] if kind == "prrt" else ["boxes", "grid", "arm", "arm", "mesh"])
    c = {"kind": kind, "scene": scene}
    if scene == "grid":
        c["size"] = _log(rng, 512, 4096)
    elif scene == "arm":
        c["links"], c["disks"] = rng.choice([5, 10, 20, 20]), rng.randint(50, 200)
    elif scene == "mesh":
        c["robot"], c["env"] = rng.choice([120, 250, 500]), rng.choice([6000, 20000, 50000])
    order = rng.choice(["reference", "surrogate"]) if scene == "arm" and c["links"] == 20 else "reference"
    if kind == "prrt":
        batch = _log(rng, 100, 8192)
        return {**c, "batch": batch, "nodes": int(batch * rng.uniform(0.5, 1.2)) + 1, "order": order}
    most = {"boxes": 1 << 20, "grid": 1 << 20, "arm": 8192, "mesh": 4096}[scene]
    n = _log(rng, 32, most)
    return {**c, "n": n, "order": order, "host": n < 256 and rng.random() < 0.5}


@functools.lru_cache(maxsize=4)
def _scene(kind, *args):
    if kind == "boxes":
        return scenes.boxes_scene()
    if kind == "grid":
        return dataclasses.replace(scenes.grid_scene(seed=4, size=args[0]), range=40.0)
    if kind == "arm":
        return scenes.arm_scene(links=args[0], ndisks=args[1])
    return scenes.se3_scene(n_env_tris=args[1], n_robot_tris=args[0])


def _scene_of(case):
    keys = {"boxes": (), "grid": ("size",), "arm": ("links", "disks"), "mesh": ("robot", "env")}[case["scene"]]
    return _scene(case["scene"], *(case[k] for k in keys))


@functools.lru_cache(maxsize=1)
def _surrogate_params():
    """Surrogate weights a program loads: trained once on the 20-link arm."""
    sc = _scene("arm", 20, 200)
    with mpt_amd.Context(0) as ctx:
        nodes = _grow(ctx, sc, 3, 2048, 3000)
        surrogate.train(ctx, sc, nodes, n_samples=1 << 15, epochs=2, seed=5, holdout=1 << 10)
        return ctx.surrogate_get()


def _grow(ctx, sc, seed, batch, nodes):
    ctx.scene(sc)
    ctx.prrt_init(sc, seed=seed, batch=batch)
    ctx.prrt_add_start(sc.start)
    ctx.prrt_run(nodes)
    return ctx.tree_read()[0]


def _uniform_states(sc, n, rng):
    q = rng.uniform(sc.lo, sc.hi, (n, sc.dim))
    if sc.metric == mpt_amd.METRIC_SE3:
        q[:, :4] = rng.normal(size=(n, 4))
        q[:, :4] /= np.linalg.norm(q[:, :4], axis=1, keepdims=True)
    return q


def _extension_edges(ctx, sc, n, seed):
    """What a planner links: valid uniform states and their nearest node of a grown tree."""
    tree = _grow(ctx, sc, seed, 4096, 3000)
    rng = np.random.default_rng(seed)
    a, b = np.zeros((0, sc.dim)), np.zeros((0, sc.dim))
    while a.shape[0] < n:
        q = _uniform_states(sc, max(4 * (n - a.shape[0]), 1024), rng)
        q = q[ctx.valid(q)][: n - a.shape[0]]
        idx, dist = ctx.knn(q, 1)
        near = tree[idx[:, 0]]
        if sc.range < INF:  # steered to the planner's range
            q = (q - near) * np.minimum(1.0, sc.range / np.maximum(dist, 1e-300)) + near
        a, b = np.concatenate([a, near]), np.concatenate([b, q])
    return a, b


def _cuda(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _mlp_params(seed):
    """He-uniform weights and zero biases, as mptg_surrogate_init draws them."""
    rng = np.random.default_rng(seed)
    out = []
    for i, o in MLP:
        b = math.sqrt(6.0 / i)
        out += [rng.uniform(-b, b, (i, o)).astype(np.float32).ravel(), np.zeros(o, np.float32)]
    return np.concatenate(out)


def _train_rows(case, seed):
    """Features in [-1, 1] with BF16 values and labels of a smooth boundary."""
    g = torch.Generator().manual_seed(seed)
    x = (torch.rand(case["rows"], 64, generator=g) * 2 - 1).to(torch.bfloat16)
    w = torch.randn(64, 2, generator=g)
    y = (torch.sin(2 * (x.float() @ w)).sum(1) + 0.3 * torch.randn(case["rows"], generator=g) > 0).float()
    return x, y


def _knn_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n, m, d = case["nodes"], case["queries"], case["dim"]
    if case["metric"] == "se3":
        pts = np.concatenate([rng.normal(size=(n + m, 4)), rng.uniform(0, 100, (n + m, 3))], axis=1)
        pts[:, :4] /= np.linalg.norm(pts[:, :4], axis=1, keepdims=True)
    else:
        pts = rng.uniform(-math.pi, math.pi, (n + m, d))
    return pts[:n], pts[n:]


def prepare(case, seed):
    kind = case["kind"]
    ctx = mpt_amd.Context(0)
    st = {"case": case, "ctx": ctx, "seed": seed}
    if kind in ("prrt", "star"):
        sc = st["scene"] = _scene_of(case)
        ctx.scene(sc)
        if case.get("order") == "surrogate":
            ctx.surrogate_set(_surrogate_params())
        # where the program keeps its trees: the last iteration ends at most a batch past the target
        rows = case["nodes"] + case["batch"]
        st["out"] = {"nodes": np.zeros((rows, sc.dim)), "parents": np.full(rows, -1, np.int32),
                     "goals": np.full(4096, -1, np.int32)}
        if kind == "star":
            st["out"]["costs"] = np.zeros(rows)
    elif kind == "link":
        sc = _scene_of(case)
        n = case["n"]
        if case["scene"] == "grid":
            ctx.scene(sc)
            a, b = scenes.grid_edges(sc, n, seed=seed)
        elif case["scene"] == "boxes":
            ctx.scene(sc)
            rng = np.random.default_rng(seed)
            a = rng.uniform(sc.lo, sc.hi, (n, 2))
            b = np.clip(a + rng.normal(size=(n, 2)) * 3.0, sc.lo, sc.hi)
        else:
            a, b = _extension_edges(ctx, sc, n, seed)
        if case["order"] == "surrogate":
            ctx.surrogate_set(_surrogate_params())
        if case["host"]:
            st["a"], st["b"] = a, b
        else:
            st["a"], st["b"] = _cuda(a), _cuda(b)
            st["verdict"] = torch.zeros(n, dtype=torch.uint8, device="cuda")
            st["checks"] = torch.zeros(n, dtype=torch.int32, device="cuda")
    elif kind == "knn":
        pts, q = _knn_inputs(case, seed)
        ctx.space(METRICS[case["metric"]], case["dim"], 50.0, 1.0)
        ctx.tree_insert(pts)
        st["q"] = _cuda(q)
        st["idx"] = torch.zeros(case["queries"], case["k"], dtype=torch.int32, device="cuda")
        st["dist"] = torch.zeros(case["queries"], case["k"], dtype=torch.float64, device="cuda")
    else:
        x, y = _train_rows(case, seed)
        st["x"], st["y"], st["params"] = x.cuda(), y.cuda(), _mlp_params(seed)
    torch.cuda.synchronize()
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind in ("prrt", "star"):
        sc = st["scene"]
        ctx.tree_clear()
        if kind == "prrt":
            ctx.prrt_init(sc, seed=st["seed"], batch=case["batch"], order=ORDERS[case["order"]])
        else:
            ctx.prrt_star_init(sc, seed=st["seed"], batch=case["batch"], k=case["k"], r_nearest=case["radius_lists"])
        ctx.prrt_add_start(sc.start)
        ctx.prrt_run(case["nodes"])
        out, got = st["out"], {}
        got["nodes"], got["parents"] = ctx.tree_read()
        got["goals"] = ctx.prrt_goals()
        if kind == "star":
            got["costs"] = ctx.prrt_costs()
        for key, v in got.items():
            out[key][:v.shape[0]] = v
        return {**out, "size": ctx.tree_size()}
    if kind == "link":
        known = case["scene"] in ("arm", "mesh")  # planner edges: both ends were validated before
        if case["host"]:
            return ctx.link(st["a"], st["b"], ORDERS[case["order"]], known)
        ctx.link_dev(st["a"].data_ptr(), st["b"].data_ptr(), case["n"], ORDERS[case["order"]], known,
                     st["verdict"].data_ptr(), st["checks"].data_ptr())
        ctx.sync()  # the program reads the verdicts on torch's stream, which the context's is not ordered with
        return st["verdict"], st["checks"]
    if kind == "knn":
        ctx.knn_dev(st["q"].data_ptr(), case["queries"], case["k"], INF, st["idx"].data_ptr(), st["dist"].data_ptr())
        ctx.sync()
        return st["idx"], st["dist"]
    ctx.surrogate_set(st["params"])
    losses = ctx.surrogate_train(st["x"].data_ptr(), st["y"].data_ptr(), case["rows"], 1, case["batch"], 2e-3)
    return ctx.surrogate_get(), losses


def work(case):
    """Inputs read once, outputs written once, and the arithmetic of the
    checks, distances or products that no exact method skips."""
    kind = case["kind"]
    if kind == "train":
        n = case["rows"]
        return {"bytes": n * 132 + 8 * MLP_MACS, "flops": 6 * MLP_MACS * n}
    if kind == "knn":
        n, m, d, k = case["nodes"], case["queries"], case["dim"], case["k"]
        # each query against the nodes it returns; every row is read once
        return {"bytes": 8 * d * (n + m) + 12 * m * k, "flops": 3 * d * m * k}
    scene = case["scene"]
    d = {"boxes": 2, "grid": 2, "arm": case.get("links", 0), "mesh": 7}[scene]
    # one edge: its waypoints' state checks
    checks, flops = {"boxes": (20, 64), "grid": (20, 4), "arm": (ARM_CHECKS, FK_FLOPS * d),
                     "mesh": (20, 18 * case.get("robot", 0))}[scene]
    scene_bytes = {"boxes": 512, "grid": case.get("size", 0) ** 2 // 8, "arm": 24 * case.get("disks", 0),
                   "mesh": 36 * (case.get("robot", 0) + case.get("env", 0))}[scene]
    if kind == "link":
        n = case["n"]
        return {"bytes": n * (16 * d + 5) + scene_bytes, "flops": n * checks * flops}
    # every node of the tree came by one free edge; PRRT* adds a list of neighbours
    n = case["nodes"]
    return {"bytes": n * (8 * d + 4) + scene_bytes, "flops": n * checks * flops * (2 if kind == "star" else 1)}


def _knn_exact(case, seed):
    n, m, d = case["nodes"], case["queries"], case["dim"]
    if n * m * d > 3e10:
        return None
    pts, q = (_cuda(x) for x in _knn_inputs(case, seed))
    out = torch.empty(m, case["k"], dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // n)
    for i in range(0, m, step):
        p = q[i:i + step]
        if case["metric"] == "se3":
            dot = torch.zeros(p.shape[0], n, dtype=torch.float64, device="cuda")
            for j in range(4):
                dot += p[:, j:j + 1] * pts[None, :, j]
            dist = 50.0 * torch.acos(dot.abs().clamp(max=1.0))
            lin = torch.zeros_like(dot)
            for j in range(4, 7):
                lin += (p[:, j:j + 1] - pts[None, :, j]) ** 2
            dist += lin.sqrt()
        else:
            dist = torch.zeros(p.shape[0], n, dtype=torch.float64, device="cuda")
            for j in range(d):
                t = p[:, j:j + 1] - pts[None, :, j]
                dist += t.abs() if case["metric"] == "l1" else t * t
            if case["metric"] == "l2":
                dist = dist.sqrt()
        v = torch.topk(dist, min(case["k"], n), dim=1, largest=False, sorted=True).values
        out[i:i + step] = v
    return None, out


def _train_exact(case, seed):
    """The same Adam steps in 64 bits on the unrounded weights."""
    x, y = _train_rows(case, seed)
    x, y = x.double().cuda(), y.double().cuda()
    flat, p, at = torch.from_numpy(_mlp_params(seed)).double().cuda(), [], 0
    for i, o in MLP:
        p.append(flat[at:at + i * o].view(i, o).clone().requires_grad_())
        p.append(flat[at + i * o:at + i * o + o].clone().requires_grad_())
        at += i * o + o
    m, v = [torch.zeros_like(t) for t in p], [torch.zeros_like(t) for t in p]
    total, batches = 0.0, case["rows"] // case["batch"]
    for t in range(batches):
        h = x[t * case["batch"]:(t + 1) * case["batch"]]
        for l in range(3):
            h = torch.relu(h @ p[2 * l] + p[2 * l + 1])
        z = (h @ p[6] + p[7])[:, 0]
        loss = torch.nn.functional.binary_cross_entropy_with_logits(z, y[t * case["batch"]:(t + 1) * case["batch"]])
        grads = torch.autograd.grad(loss, p)
        total += float(loss.detach())
        with torch.no_grad():
            for k, g in enumerate(grads):
                m[k] = 0.9 * m[k] + 0.1 * g
                v[k] = 0.999 * v[k] + 0.001 * g * g
                step = (m[k] / (1 - 0.9 ** (t + 1))) / ((v[k] / (1 - 0.999 ** (t + 1))).sqrt() + 1e-8)
                p[k] -= 2e-3 * step
    return torch.cat([t.detach().reshape(-1) for t in p]), torch.tensor([total / batches], dtype=torch.float64)


def exact(case, seed):
    """64-bit values of the computed numbers.  Trees, costs and verdicts are
    decided step by step and have no closed form: None."""
    if case["kind"] == "knn":
        return _knn_exact(case, seed)
    if case["kind"] == "train":
        return _train_exact(case, seed)
    return None
