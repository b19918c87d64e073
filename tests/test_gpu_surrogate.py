"""GPU surrogate: forward/backward kernels against the CPU oracle, training on
exact-checker labels, and the surrogate-ordered link() — same verdicts as the
reference order, check counts equal to the oracle's count for the GPU's own
scores, fewer checks in total."""
import math
import sys

import numpy as np
import pytest

import mpt_amd
import oracle
from conftest import GPU_ITER_CAP
from mpt_amd import scenes

pytestmark = pytest.mark.gpu

NP = 41473
OFF = {"W1": 0, "b1": 8192, "W2": 8320, "b2": 24704, "W3": 24832, "b3": 41216, "w4": 41344, "b4": 41472}


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _bits_to_f32(u16):
    return (u16.astype(np.uint32) << 16).view(np.float32)


def _net(seed):
    rng = np.random.default_rng(seed)
    p = np.zeros(NP, dtype=np.float32)
    for w, b, fan in (("W1", "b1", 64), ("W2", "b2", 128), ("W3", "b3", 128), ("w4", "b4", 128)):
        p[OFF[w]:OFF[b]] = rng.uniform(-1, 1, OFF[b] - OFF[w]) * math.sqrt(6 / fan)
    p[OFF["b1"]:OFF["W2"]] = rng.normal(0, 0.1, 128)
    p[OFF["b2"]:OFF["W3"]] = rng.normal(0, 0.1, 128)
    p[OFF["b3"]:OFF["w4"]] = rng.normal(0, 0.1, 128)
    p[OFF["b4"]] = 0.05
    return p


def _data(seed, n):
    rng = np.random.default_rng(seed)
    X = oracle.bf16(rng.normal(0, 1, (n, 64)).astype(np.float32))
    y = (rng.uniform(size=n) < 0.4).astype(np.float32)
    return X, y


def _tensor_slices():
    return [(k, OFF[k], OFF[n]) for k, n in (("W1", "b1"), ("b1", "W2"), ("W2", "b2"), ("b2", "W3"), ("W3", "b3"),
                                              ("b3", "w4"), ("w4", "b4"))] + [("b4", OFF["b4"], NP)]


def test_loss_grad_parity(ctx_factory):
    _say("surrogate loss/grad parity")
    ctx = ctx_factory()
    p = _net(11)
    X, y = _data(12, 512)
    ctx.surrogate_set(p)
    dX, dy = ctx.to_device(X), ctx.to_device(y)
    loss, g = ctx.surrogate_loss_grad(dX.ptr, dy.ptr, 512)
    ol, og, _ = oracle.mlp_loss_grad(p, X, y)
    assert abs(loss - ol) <= 1e-4 * abs(ol)
    for name, a, b in _tensor_slices():
        gg, oo = g[a:b].astype(np.float64), og[a:b].astype(np.float64)
        # FP32 accumulation order and rare BF16 rounding flips differ
        assert np.linalg.norm(gg - oo) <= 1e-2 * np.linalg.norm(oo) + 1e-7, name
        if b - a > 1:
            assert float(np.dot(gg, oo)) >= 0.9999 * np.linalg.norm(gg) * np.linalg.norm(oo), name


def test_forward_parity(ctx_factory):
    _say("surrogate forward parity")
    ctx = ctx_factory()
    p = _net(13)
    X, y = _data(14, 1000)  # not a multiple of 16: padded inside
    ctx.surrogate_set(p)
    dX = ctx.to_device(X)
    dz = ctx.array(1000, np.float32)
    ctx.surrogate_forward(dX.ptr, 1000, dz.ptr)
    _, _, oz = oracle.mlp_loss_grad(p, X, y)
    z = dz.numpy()
    assert np.allclose(z, oz, rtol=2e-2, atol=2e-2)
    assert np.corrcoef(z, oz)[0, 1] > 0.9999


def test_adam_step_parity(ctx_factory):
    _say("surrogate adam parity")
    ctx = ctx_factory()
    p = _net(15)
    X, y = _data(16, 256)
    ctx.surrogate_set(p)
    dX, dy = ctx.to_device(X), ctx.to_device(y)
    _, g = ctx.surrogate_loss_grad(dX.ptr, dy.ptr, 256)
    ctx.surrogate_set(p)
    ctx.surrogate_train(dX.ptr, dy.ptr, 256, epochs=1, batch=256, lr=1e-3)
    p1 = ctx.surrogate_get()
    e1, _, _ = oracle.adam_step(p, np.zeros(NP), np.zeros(NP), g, lr=1e-3, t=1)
    assert np.mean(np.abs(p1 - e1) <= 1e-6) > 0.999


@pytest.mark.parametrize("n", [16, 32, 48, 256, 4112, 16432])
def test_pass_sizes_parity(ctx_factory, n):
    """A half tile of rows, whole tiles, tiles that end half full, a sum's
    unrolled chunks (256 rows) with and without a rest, and more tiles than
    blocks (16384 rows), from aligned rows and from rows the pass
    kernel has to copy (2-byte offset): loss and gradient against the oracle
    with test_loss_grad_parity's bounds, and the logits of the same rows."""
    _say("surrogate pass", n)
    ctx = ctx_factory()
    p = _net(18)
    X, y = _data(19, n)
    ctx.surrogate_set(p)
    ol, og, oz = oracle.mlp_loss_grad(p, X, y)
    dy, dz = ctx.to_device(y), ctx.array(n, np.float32)
    for shift in (0, 1):
        dX = ctx.to_device(np.concatenate([np.zeros(shift, np.uint16), X.ravel()]))
        ptr = dX.ptr + 2 * shift
        loss, g = ctx.surrogate_loss_grad(ptr, dy.ptr, n)
        assert abs(loss - ol) <= 1e-4 * abs(ol)
        for name, a, b in _tensor_slices():
            gg, oo = g[a:b].astype(np.float64), og[a:b].astype(np.float64)
            assert np.linalg.norm(gg - oo) <= 1e-2 * np.linalg.norm(oo) + 1e-7, (shift, name)
        ctx.surrogate_forward(ptr, n, dz.ptr)
        assert np.allclose(dz.numpy(), oz, rtol=2e-2, atol=2e-2), shift
    # the sums' order is fixed: the same bits every time
    l2, g2 = ctx.surrogate_loss_grad(ptr, dy.ptr, n)
    assert l2 == loss and np.array_equal(g2, g)


def test_features_match_forward_kinematics(ctx_factory):
    _say("surrogate features")
    ctx = ctx_factory()
    sc = scenes.arm_scene()
    ctx.scene(sc)
    rng = np.random.default_rng(17)
    q = rng.uniform(-math.pi, math.pi, (500, 20))
    f = ctx.array((500, 64), np.uint16)
    dq = ctx.to_device(q)
    ctx.surrogate_features(dq.ptr, 500, f.ptr)
    got = _bits_to_f32(f.numpy())
    ang = np.cumsum(q, axis=1)
    x = np.cumsum(sc.lengths * np.cos(ang), axis=1) / sc.lengths.sum()
    yy = np.cumsum(sc.lengths * np.sin(ang), axis=1) / sc.lengths.sum()
    exp = np.zeros((500, 64))
    exp[:, 0:40:2], exp[:, 1:40:2] = x, yy
    exp[:, 40:64:2], exp[:, 41:64:2] = np.cos(ang[:, :12]), np.sin(ang[:, :12])
    assert np.allclose(got, exp, rtol=1e-2, atol=2e-3)


def _valid_states(ctx, sc, n, seed):
    rng = np.random.default_rng(seed)
    out = []
    while sum(len(o) for o in out) < n:
        q = rng.uniform(sc.lo, sc.hi, (4 * n, sc.dim))
        out.append(q[ctx.valid(q)])
    return np.concatenate(out)[:n]


def _auc(scores, labels):
    order = np.argsort(scores, kind="stable")
    ranks = np.empty(len(scores))
    ranks[order] = np.arange(1, len(scores) + 1)
    pos = labels > 0.5
    npos, nneg = pos.sum(), (~pos).sum()
    return (ranks[pos].sum() - npos * (npos + 1) / 2) / (npos * nneg)


@pytest.fixture(scope="module")
def trained(ctx_factory):
    """Arm scene + a surrogate trained on 2^17 exact-checker labels."""
    ctx = ctx_factory()
    sc = scenes.arm_scene()
    ctx.scene(sc)
    n = 1 << 17
    a = _valid_states(ctx, sc, n, 21)
    b = np.clip(a + np.random.default_rng(22).normal(0, 0.8, a.shape), -math.pi, math.pi)
    feat = ctx.array((n, 64), np.uint16)
    lab = ctx.array(n, np.float32)
    da, db = ctx.to_device(a), ctx.to_device(b)
    ctx.surrogate_samples(da.ptr, db.ptr, n, 23, feat.ptr, lab.ptr)
    ctx.surrogate_init(24)
    losses = ctx.surrogate_train(feat.ptr, lab.ptr, n, epochs=6, batch=1024, lr=2e-3)
    return ctx, sc, losses, feat, lab


def test_training_learns_collision_labels(trained):
    _say("surrogate training")
    ctx, sc, losses, _, lab = trained
    _say("epoch losses", losses)
    assert losses[-1] < 0.85 * losses[0]
    m = 1 << 14
    a = _valid_states(ctx, sc, m, 31)
    b = np.clip(a + np.random.default_rng(32).normal(0, 0.8, a.shape), -math.pi, math.pi)
    feat = ctx.array((m, 64), np.uint16)
    y = ctx.array(m, np.float32)
    da, db = ctx.to_device(a), ctx.to_device(b)
    ctx.surrogate_samples(da.ptr, db.ptr, m, 33, feat.ptr, y.ptr)
    z = ctx.array(m, np.float32)
    ctx.surrogate_forward(feat.ptr, m, z.ptr)
    yy = y.numpy()
    auc = _auc(z.numpy(), yy)
    _say("held-out AUC", auc, "positives", float(yy.mean()))
    assert auc > 0.8


def test_surrogate_order_parity_and_savings(trained):
    _say("surrogate-ordered link")
    ctx, sc, _, _, _ = trained
    m = 512
    a = _valid_states(ctx, sc, m, 41)
    b = _valid_states(ctx, sc, m, 42)
    v_ref, c_ref = ctx.link(a, b, mpt_amd.ORDER_REFERENCE, True)
    v_sur, c_sur = ctx.link(a, b, mpt_amd.ORDER_SURROGATE, True)
    assert np.array_equal(v_ref, v_sur)
    ov, oc = oracle.Oracle(sc).link(a, b, known_valid=True, threads=16)
    assert np.array_equal(v_ref, ov) and np.array_equal(c_ref, oc)
    scores = ctx.array((m, 512), np.float32)
    da, db = ctx.to_device(a), ctx.to_device(b)
    ctx.surrogate_score_edges(da.ptr, db.ptr, m, scores.ptr)
    sc_np = scores.numpy()
    o = oracle.Oracle(sc)
    # the surrogate order: the 4 best-scored waypoints of the top 4
    # bisection levels (the picks), then every other waypoint in
    # reference order
    for e in range(0, m, 2):
        W = len(o.waypoints(a[e], b[e]))
        assert c_sur[e] == o.checks_in_score_order(a[e], b[e], sc_np[e, :W], known_valid=True, lead=0,
                                                   top_levels=4, picks=4), e
    # fused scores == generic forward on the same waypoints, up to the BF16
    # rounding of features built from FP32-interpolated waypoints
    zs, ss = [], []
    for e in range(0, 24):
        wp = o.waypoints(a[e], b[e])
        W = len(wp)
        f = ctx.array((W, 64), np.uint16)
        dwp = ctx.to_device(wp)
        ctx.surrogate_features(dwp.ptr, W, f.ptr)
        z = ctx.array(W, np.float32)
        ctx.surrogate_forward(f.ptr, W, z.ptr)
        zs.append(z.numpy())
        ss.append(sc_np[e, :W])
    zs, ss = np.concatenate(zs), np.concatenate(ss)
    assert np.allclose(zs, ss, rtol=0.05, atol=0.05)
    assert np.corrcoef(zs, ss)[0, 1] > 0.999
    coll = ~v_ref
    _say("colliding", int(coll.sum()), "checks ref", int(c_ref[coll].sum()), "sur", int(c_sur[coll].sum()))
    assert c_sur[coll].sum() < 0.8 * c_ref[coll].sum()
    assert np.array_equal(c_sur[~coll], c_ref[~coll])  # valid edges check everything in both orders


def test_planner_with_surrogate_order_grows_the_oracle_tree(trained):
    """Check order never changes a verdict, so the surrogate-ordered planner
    grows exactly the reference-order tree (and the oracle's)."""
    _say("surrogate-ordered planner")
    ctx, sc, _, _, _ = trained
    ctx.tree_clear()
    ctx.prrt_init(sc, 13, 256, order=mpt_amd.ORDER_SURROGATE)
    ctx.prrt_add_start(sc.start)
    st = ctx.prrt_run(400, GPU_ITER_CAP)
    gn, gp = ctx.tree_read()
    on, op, og, ost = oracle.Oracle(sc).prrt(13, 256, 400)
    assert np.array_equal(gn, on) and np.array_equal(gp, op)
    assert st["link_calls"] == ost["link_calls"] and st["link_ok"] == ost["link_ok"]
    assert st["valid_calls"] < ost["valid_calls"]  # surrogate order: fewer checks than the reference order


def test_surrogate_planner_in_graph_mode_equals_step_by_step(trained):
    """Captured iterations with the surrogate order (score, rank, head, tail
    kernels inside the graph) grow the step-by-step tree with the same
    counters, check counts included."""
    _say("surrogate planner graph")
    ctx, sc, _, _, _ = trained
    res = []
    for g in (0, 4):
        ctx.tree_clear()
        ctx.prrt_init(sc, 14, 512, order=mpt_amd.ORDER_SURROGATE)
        ctx.prrt_graph(g)
        ctx.prrt_add_start(sc.start)
        st = ctx.prrt_run(1200, GPU_ITER_CAP)
        gn, gp = ctx.tree_read()
        res.append((gn, gp, st))
    ctx.prrt_graph(0)
    (an, ap, ast), (bn, bp, bst) = res
    assert ast["graph_launches"] == 0 and bst["graph_launches"] > 0
    assert np.array_equal(an, bn) and np.array_equal(ap, bp)
    for key in ("iterations", "samples", "zero_dist", "invalid_states", "link_calls", "link_ok", "valid_calls",
                "goals"):
        assert ast[key] == bst[key], key
