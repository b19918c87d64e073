"""Neighbour lists beyond 32 entries and without a length limit, and PRRT*
with the reference's neighbour rules.

* k-nearest with k = 33..64 (the reference's k = ceil(kRRG ln(n + 1)) is 48 at
  10^6 nodes in 7-D, src/mpt/impl/rrg_rewire_neighbors.hpp:53-67);
* every node within a radius (nigh's nearest(nbh, q, SIZE_MAX, r),
  rrg_rewire_neighbors.hpp:124-128) through mptg_rnn's count-then-fill;
* PRRT* with rewire_r_nearest (lists of any length) and with the default k
  formula, against the oracle, and the default PRRTStar<> growing 10^5 nodes in SE(3) (7
  coordinates)."""
import dataclasses
import math
import sys

import numpy as np
import pytest

import mpt_amd
import oracle
from conftest import GPU_ITER_CAP
from mpt_amd import scenes

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _plain(metric, dim, w_so3=1.0, w_l2=1.0):
    return scenes.Scene(metric=metric, dim=dim, kind=scenes.SCENE_NONE, link_mode=scenes.LINK_DMV, link_param=1.0,
                        lo=np.zeros(dim), hi=np.ones(dim), start=np.zeros(dim), goal=np.zeros(dim),
                        w_so3=w_so3, w_l2=w_l2)


def _se3_states(rng, n):
    qu = rng.normal(size=(n, 4))
    qu /= np.linalg.norm(qu, axis=1, keepdims=True)
    return np.concatenate([qu, rng.uniform(0, 100, (n, 3))], axis=1)


@pytest.mark.parametrize("metric,dim,k,n", [
    (scenes.METRIC_L2, 7, 48, 6000), (scenes.METRIC_L1, 20, 64, 4000), (scenes.METRIC_L2, 2, 33, 3000),
    (scenes.METRIC_SE3, 7, 64, 2000),
])
def test_knn_large_k_parity(ctx_factory, metric, dim, k, n):
    _say("knn large k", metric, dim, k)
    ctx = ctx_factory()
    rng = np.random.default_rng(100 + k)
    w = (50.0, 1.0) if metric == scenes.METRIC_SE3 else (1.0, 1.0)
    pts = _se3_states(rng, n) if metric == scenes.METRIC_SE3 else rng.uniform(-math.pi, math.pi, (n, dim))
    pts[n // 2] = pts[n // 3]  # duplicates: ties by index
    q = _se3_states(rng, 500) if metric == scenes.METRIC_SE3 else rng.uniform(-math.pi, math.pi, (500, dim))
    ctx.space(metric, dim, *w)
    ctx.tree_insert(pts)
    o = oracle.Oracle(_plain(metric, dim, *w))
    for radius in (math.inf, None):
        if radius is None:  # a radius that cuts some lists short
            radius = float(np.median(o.knn(pts, q[:50], k, threads=16)[1][:, k // 2]))
        gi, gd = ctx.knn(q, k, radius=radius)
        oi, od = o.knn(pts, q, k, radius=radius, threads=16)
        assert np.array_equal(gi, oi) and np.array_equal(gd, od), radius


@pytest.mark.parametrize("metric,dim", [(scenes.METRIC_L2, 2), (scenes.METRIC_L1, 20), (scenes.METRIC_L2, 7),
                                        (scenes.METRIC_SE3, 7)])
def test_rnn_every_node_within_radius(ctx_factory, metric, dim):
    _say("rnn", metric, dim)
    ctx = ctx_factory()
    rng = np.random.default_rng(200 + dim)
    w = (50.0, 1.0) if metric == scenes.METRIC_SE3 else (1.0, 1.0)
    n = 9000  # three tree chunks
    pts = _se3_states(rng, n) if metric == scenes.METRIC_SE3 else rng.uniform(-math.pi, math.pi, (n, dim))
    pts[100:120] = pts[5]  # ties at equal distance keep ascending ids
    q = _se3_states(rng, 300) if metric == scenes.METRIC_SE3 else rng.uniform(-math.pi, math.pi, (300, dim))
    q[0] = pts[5]
    ctx.space(metric, dim, *w)
    ctx.tree_insert(pts)
    o = oracle.Oracle(_plain(metric, dim, *w))
    typical = float(np.median(o.knn(pts, q[:30], 40, threads=16)[1][:, -1]))
    for radius in (0.0, typical, 1e300):
        off, gi, gd = ctx.rnn(q, radius, cap=100)  # small first guess: the call retries with the count
        assert off[0] == 0 and (np.diff(off) >= 0).all()
        oi, od = o.knn(pts, q, n, radius=radius, threads=16)
        for i in range(q.shape[0]):
            sel = oi[i] >= 0
            assert np.array_equal(gi[off[i]:off[i + 1]], oi[i][sel]), (radius, i)
            assert np.array_equal(gd[off[i]:off[i + 1]], od[i][sel]), (radius, i)
        if radius == 1e300:
            assert off[-1] == n * q.shape[0]
    off, gi, gd = ctx.rnn(np.zeros((0, dim)), 1.0)
    assert off.tolist() == [0] and gi.size == 0


def _star(ctx, sc, seed, batch, target, k=20, r_nearest=False, factor=1.1, max_iters=1 << 30):
    ctx.scene(sc)
    ctx.tree_clear()
    ctx.prrt_star_init(sc, seed, batch, k=k, rewire_factor=factor, r_nearest=r_nearest)
    ctx.prrt_add_start(sc.start)
    st = ctx.prrt_run(target, min(max_iters, GPU_ITER_CAP))
    gn, gp = ctx.tree_read()
    return gn, gp, ctx.prrt_costs(), st


@pytest.mark.parametrize("name,batch,target", [("boxes", 1, 600), ("boxes", 64, 3000), ("arm", 128, 500),
                                               ("se3", 256, 1500)])
def test_prrt_star_r_nearest_equals_oracle(ctx_factory, name, batch, target):
    _say("prrt* r-nearest", name, batch)
    sc = {"boxes": scenes.boxes_scene, "arm": scenes.arm_scene, "se3": scenes.se3_scene}[name]()
    gn, gp, gc, st = _star(ctx_factory(), sc, 31, batch, target, r_nearest=True)
    on, op, oc, og, ost, oss = oracle.Oracle(sc).prrt_star(31, batch, target, k=-1)
    assert np.array_equal(gn, on) and np.array_equal(gp, op) and np.array_equal(gc, oc)
    for key in ("rewire_tests", "rewires", "parent_changes", "deferred"):
        assert st[key] == oss[key], key
    assert st["cp_links"] == oss["spec_cp"]
    assert st["rw_links"] == oss["spec_rw"] + st["rw_late"] and st["rw_late"] >= oss["deferred"]
    if name == "boxes":
        assert st["rewires"] > 0


@pytest.mark.parametrize("name,batch,target,factor", [("boxes", 64, 4000, 2.5), ("se3", 128, 1200, 12.0)])
def test_prrt_star_r_nearest_long_lists(ctx_factory, name, batch, target, factor):
    """A larger rewire factor puts hundreds of nodes in every list (about 230
    in the 2-D case, 450 in SE(3)): the lists are not cut, and the walks over
    several 64-entry pages, their rewires and deferred edges equal the
    oracle's."""
    _say("prrt* r-nearest long lists", name)
    sc = {"boxes": scenes.boxes_scene, "se3": scenes.se3_scene}[name]()
    gn, gp, gc, st = _star(ctx_factory(), sc, 32, batch, target, r_nearest=True, factor=factor)
    on, op, oc, og, ost, oss = oracle.Oracle(sc).prrt_star(32, batch, target, k=-1, rewire_factor=factor)
    assert np.array_equal(gn, on) and np.array_equal(gp, op) and np.array_equal(gc, oc)
    for key in ("rewire_tests", "rewires", "parent_changes", "deferred"):
        assert st[key] == oss[key], key
    assert st["cp_links"] == oss["spec_cp"]
    assert st["rw_links"] == oss["spec_rw"] + st["rw_late"] and st["rw_late"] >= oss["deferred"]
    assert st["rewire_tests"] > 200 * (len(gn) - 1) and st["rewires"] > 500 and st["deferred"] > 0


def test_prrt_star_reference_k_formula_se3(ctx_factory):
    """k = ceil(kRRG ln(n + 1)) with the SE(3) space's dimension 6."""
    _say("prrt* k formula se3")
    sc = scenes.se3_scene()
    gn, gp, gc, st = _star(ctx_factory(), sc, 33, 256, 2500, k=0)
    on, op, oc, og, ost, oss = oracle.Oracle(sc).prrt_star(33, 256, 2500, k=0)
    assert np.array_equal(gn, on) and np.array_equal(gp, op) and np.array_equal(gc, oc)
    assert oracle.lib().orc_star_k(0, 1.1, 6, 2500) == 28


def test_default_prrt_star_grows_1e5_nodes_in_se3(ctx_factory):
    """The default PRRTStar<> (k formula, 41 neighbours at 10^5 nodes in
    SE(3)) grows a tree of 10^5 nodes; its costs add up along the edges and
    every node hangs off the start."""
    _say("prrt* default to 1e5 nodes")
    sc = scenes.se3_scene()
    ctx = ctx_factory()
    gn, gp, gc, st = _star(ctx, sc, 34, 4096, 100_000, k=0)
    assert len(gn) >= 100_000 and oracle.lib().orc_star_k(0, 1.1, 6, len(gn) - 1) >= 40
    o = oracle.Oracle(sc)
    d = np.array([o.distance(gn[gp[i]], gn[i]) for i in range(1, len(gn))])
    assert np.allclose(gc[1:], gc[gp[1:]] + d, rtol=1e-12, atol=1e-9)
    assert gp[0] == -1 and ((gp[1:] >= 0) & (gp[1:] < len(gn))).all()
    anc = gp.copy()  # pointer doubling: every node reaches the start (no cycle)
    anc[0] = 0
    for _ in range(20):
        anc = anc[anc]
    assert (anc == 0).all()
    assert st["rewires"] > 0


# k = 1 (knn_one.hip): trees of less than a block's rows and one row either
# side of them, odd counts of queries for 1, 4, 8 and 16 per block, a larger
# tree that few queries leave to the scan
@pytest.mark.parametrize("scale", [1.0, 1e25], ids=["plain", "beyond-fp32-squares"])
@pytest.mark.parametrize("metric,dim,n,nq", [
    (scenes.METRIC_L2, 1, 1, 1), (scenes.METRIC_L1, 2, 255, 7), (scenes.METRIC_L2, 2, 256, 1023),
    (scenes.METRIC_L2, 2, 1025, 1025), (scenes.METRIC_L2, 2, 5000, 4097), (scenes.METRIC_L1, 3, 2049, 2049),
    (scenes.METRIC_L2, 4, 511, 1024), (scenes.METRIC_L1, 5, 513, 2050), (scenes.METRIC_L2, 6, 3000, 40),
    (scenes.METRIC_L2, 7, 65535, 65), (scenes.METRIC_L1, 8, 4100, 2055), (scenes.METRIC_L2, 3, 65537, 3),
])
def test_knn_nearest_equals_oracle(ctx_factory, metric, dim, n, nq, scale):
    _say("knn nearest", metric, dim, n, nq, scale)
    ctx = ctx_factory()
    ctx.tune_set(knn_grid=0)
    rng = np.random.default_rng(dim * 1000 + n)
    pts = rng.uniform(-2, 2, (n, dim)) * scale
    pts[n // 2:n // 2 + 3] = pts[0]  # equal distances: the lowest id
    pts[256::256][:3] = pts[0]  # and some that fall to the same lane
    q = rng.uniform(-2.5, 2.5, (nq, dim)) * scale
    q[0] = pts[0]
    ctx.space(metric, dim)
    ctx.tree_insert(pts)
    o = oracle.Oracle(_plain(metric, dim))
    some = np.unique(np.concatenate([[0, nq - 1], rng.integers(0, nq, 400)]))
    for radius in (math.inf, 0.1 * scale):
        gi, gd = ctx.knn(q, 1, radius=radius)
        oi, od = o.knn(pts, q[some], 1, radius=radius, threads=8)
        assert np.array_equal(gi[some], oi) and np.array_equal(gd[some], od), radius


@pytest.mark.parametrize("metric,dim,n,nq", [
    (scenes.METRIC_L1, 8, 700, 16385), (scenes.METRIC_L1, 8, 2050, 16383), (scenes.METRIC_L1, 8, 40001, 841),
    (scenes.METRIC_L1, 8, 65537, 8193), (scenes.METRIC_L2, 8, 65537, 8193), (scenes.METRIC_L2, 1, 100001, 8193),
    (scenes.METRIC_L1, 5, 100001, 8193), (scenes.METRIC_L1, 3, 131073, 8193), (scenes.METRIC_L2, 6, 262145, 8193),
    (scenes.METRIC_L1, 20, 30001, 1025),
])
@pytest.mark.parametrize("spread", [1.0, 1.3], ids=["inside", "beyond-the-tree"])
def test_knn_nearest_routes_agree(ctx_factory, metric, dim, n, nq, spread):
    """k = 1 on both sides of the lines between a block per query and the
    scans (with and without the byte prefilter): the same ids and distances,
    the oracle's.  Queries a little and far outside the tree's box, where the
    byte rows are clamped, and past where they are used."""
    _say("knn nearest routes", metric, dim, n, nq, spread)
    ctx = ctx_factory()
    rng = np.random.default_rng(dim * 1000 + n)
    pts = rng.uniform(-2, 2, (n, dim))
    pts[n // 2:n // 2 + 3] = pts[0]
    q = rng.uniform(-1.9 * spread, 1.9 * spread, (nq, dim))
    if spread > 1.0:
        for i, far in enumerate((1.1, 3.0, 1e3, 2.0 ** 19, 2.0 ** 22, 1e17)):
            q[1 + i] *= far
            q[100 + i, dim - 1] *= far  # one coordinate alone
    q[0] = pts[0]
    ctx.space(metric, dim)
    ctx.tree_insert(pts)
    o = oracle.Oracle(_plain(metric, dim))
    some = np.unique(np.concatenate([np.arange(7), np.arange(100, 106), [nq - 1], rng.integers(0, nq, 100)]))
    oi, od = o.knn(pts, q[some], 1, radius=math.inf, threads=8)
    got = []
    for q8 in (1, 0):
        ctx.tune_set(knn_grid=0, knn_q8=q8)
        got.append(ctx.knn(q, 1))
        assert np.array_equal(got[-1][0][some], oi) and np.array_equal(got[-1][1][some], od), q8
    few = ctx.knn(q[:300], 1)
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    assert np.array_equal(got[0][0][:300], few[0]) and np.array_equal(got[0][1][:300], few[1])


@pytest.mark.parametrize("metric,dim", [(scenes.METRIC_L2, 1), (scenes.METRIC_L2, 2), (scenes.METRIC_L1, 3),
                                        (scenes.METRIC_L2, 7), (scenes.METRIC_L1, 8)])
@pytest.mark.parametrize("nq", [3, 1025, 4099])
@pytest.mark.parametrize("places", [1, 9, 4000])
def test_knn_nearest_of_many_at_one_place(ctx_factory, metric, dim, nq, places):
    """Thousands of nodes at a few points, more pairs under the threshold than
    a block lists: the lowest id of the nearest point, the oracle's, for
    queries at the points, beside them, out of the radius and at infinity."""
    _say("knn crowded", metric, dim, nq, places)
    ctx = ctx_factory()
    rng = np.random.default_rng(dim + places)
    n = 5003
    pts = rng.uniform(-2, 2, (places, dim))[rng.integers(0, places, n)]
    q = rng.uniform(-2.5, 2.5, (nq, dim))
    q[::5] = pts[rng.integers(0, n, len(q[::5]))]
    q[2, 0] = math.inf  # every node at the one distance
    ctx.space(metric, dim)
    ctx.tree_insert(pts)
    o = oracle.Oracle(_plain(metric, dim))
    for radius in (math.inf, 0.3, 0.0):
        gi, gd = ctx.knn(q, 1, radius=radius)
        oi, od = o.knn(pts, q, 1, radius=radius, threads=8)
        assert np.array_equal(gi, oi) and np.array_equal(gd, od), radius


# wave lists (knn_wave.hip): rows shorter than a wave, one row either side of
# a wave's 64 nodes, the tree sizes where a query gets 4 and 16 waves, and
# enough queries (an odd count) for four per wave
@pytest.mark.parametrize("metric,dim,k,n,nq", [
    (scenes.METRIC_L2, 2, 2, 1, 3), (scenes.METRIC_L2, 2, 20, 63, 100), (scenes.METRIC_L1, 3, 64, 64, 70),
    (scenes.METRIC_L2, 7, 64, 65, 70), (scenes.METRIC_L1, 1, 5, 1023, 64), (scenes.METRIC_L2, 12, 33, 1024, 1),
    (scenes.METRIC_L2, 2, 45, 4095, 1000), (scenes.METRIC_L1, 20, 20, 4097, 33), (scenes.METRIC_L2, 16, 7, 5000, 40),
    (scenes.METRIC_L2, 2, 20, 900, 32769), (scenes.METRIC_L1, 8, 11, 700, 40001), (scenes.METRIC_L2, 10, 3, 300, 33001),
])
def test_knn_wave_lists_equal_oracle(ctx_factory, metric, dim, k, n, nq):
    _say("knn wave lists", metric, dim, k, n, nq)
    ctx = ctx_factory()
    rng = np.random.default_rng(dim * 1000 + n)
    pts = rng.uniform(-2, 2, (n, dim))
    pts[n // 2:n // 2 + 3] = pts[0]  # equal distances: ascending ids
    q = rng.uniform(-2.5, 2.5, (nq, dim))
    q[0] = pts[0]
    ctx.space(metric, dim)
    ctx.tree_insert(pts)
    o = oracle.Oracle(_plain(metric, dim))
    some = np.unique(np.concatenate([[0, nq - 1], rng.integers(0, nq, 400)]))
    for radius in (math.inf, 1.0):
        gi, gd = ctx.knn(q, k, radius=radius)
        oi, od = o.knn(pts, q[some], k, radius=radius, threads=8)
        assert np.array_equal(gi[some], oi) and np.array_equal(gd[some], od), radius
