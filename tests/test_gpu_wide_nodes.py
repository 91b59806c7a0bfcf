"""The 4-wide quantized traversal hierarchy against the oracle's binary
traversal: geometry whose nodes are flat, translated far from the origin
against the size of its triangles, nested deeply, tiny (one to five
primitives, so that slots of a node stay unused), and leaf limits that keep
every subtree split, none, or the default ones. Ids, distances and barycentrics
bit for bit: the quantized boxes only cull, what is tested is decided by the
leaves' full-precision boxes."""
import numpy as np
import pytest

import scene_util as U
from mufflon_amd import scenes as S

pytestmark = pytest.mark.gpu


def _grid(n):
    """A horizontal sheet of 2 n^2 triangles: nodes without extent in y."""
    v, _, _, t = S.grid_mesh(np.zeros((n + 1, n + 1), np.float32), 1.0 / n, 1.0)
    return v, t


def _nested(levels):
    """Triangles that halve one axis after the other towards the origin: a
    chain of `levels` Morton splits whose boxes all hold the origin's corner."""
    v = []
    s = np.array([1.0, 1.0, 1.0])
    for k in range(levels):
        v += [[0, 0, s[2]], [s[0], 0, 0.3 * s[2]], [0, s[1], 0.1 * s[2]]]
        s[k % 3] *= 0.5
    return np.array(v, np.float32), np.arange(3 * levels, dtype=np.uint32).reshape(-1, 3)


def _geometry(name):
    if name == "grid":
        return _grid(40)
    if name == "nested":
        return _nested(60)
    if name.startswith("soup"):
        return S.random_triangle_soup(int(name[4:]), seed=9, mu=-2.0)
    v, t = S.random_triangle_soup(20000, seed=4, mu=-4.0)
    return (v + np.float32(16.0) if name == "translated" else v), t


@pytest.mark.parametrize("name,limit", [("grid", 16), ("nested", 1), ("nested", 16), ("soup2", 16), ("soup3", 16),
                                        ("soup5", 1), ("soup17", 16), ("translated", 16), ("dense", 0), ("dense", 1),
                                        ("dense", 1000)])
def test_wide_traversal_matches_oracle(hip_ctx, oracle, name, limit):
    print("wide nodes %s limit %d" % (name, limit), flush=True)
    v, t = _geometry(name)
    hip_ctx.set_traversal_leaf_limit(limit)
    try:
        lod = hip_ctx.lod_create(v, t)
        hip_ctx.lbvh_build(lod)
    finally:
        hip_ctx.set_traversal_leaf_limit(16)
    rng = np.random.default_rng(3)
    lo, hi = v.min(0).astype(np.float64), v.max(0).astype(np.float64)
    n = 20000
    o = lo + (hi - lo + 1e-3) * rng.uniform(-1.5, 2.5, (n, 3))
    target = v[t[rng.integers(0, len(t), n)]].mean(1) + (hi - lo) * rng.normal(scale=0.01, size=(n, 3))
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = o
    rays[:, 3] = S.MAX_SCENE_SIZE
    d = target - o
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    for il, w in ((np.zeros(1, np.int32), S.IDENTITY34.reshape(1, 12)),
                  (np.zeros(3, np.int32), np.concatenate([S.IDENTITY34.reshape(1, 12), U.random_transforms(2, 8)]))):
        sc = hip_ctx.scene_create(np.full(len(il), lod, np.int32), w)
        oscene, _ = U.oracle_scene(oracle, [(v, t)], il, w)
        gt, gi, gp, gb, st = hip_ctx.trace_closest(sc, rays)
        ot, oi, op, ob = oracle.trace_closest(oscene, rays)
        assert (st == 0).all()
        assert np.array_equal(gi, oi) and np.array_equal(gp, op)
        assert np.array_equal(gt.view(np.uint32), ot.view(np.uint32))
        hit = oi >= 0
        assert hit.any()
        assert np.array_equal(gb[hit].view(np.uint32), ob[hit].view(np.uint32))
        assert np.array_equal(hip_ctx.trace_any(sc, rays), oracle.trace_any(oscene, rays))


def test_full_stack(hip_ctx, oracle):
    """45 instances that halve one axis after the other towards the origin, a
    chain of the instance level: rays to the origin enter the inner side first
    and leave two entries a level behind, more than the 64 of the wide stack, so
    they are handed to the reference traversal. Others stay below."""
    v, t = S.random_triangle_soup(300, seed=8, mu=-1.5)
    v = np.clip(v, 0.0, 1.0).astype(np.float32)
    v[:6] = [[0, 0, 0], [1, 1, 1], [1, 0, 1], [0, 1, 0], [1, 0, 0], [0, 1, 1]]
    s = np.ones(3)
    w = []
    for k in range(45):
        w.append(np.array([1 / s[0], 0, 0, 0, 0, 1 / s[1], 0, 0, 0, 0, 1 / s[2], 0], np.float32))
        s[k % 3] *= 0.5
    lod = hip_ctx.lod_create(v, t)
    hip_ctx.lbvh_build(lod)
    il = np.zeros(45, np.int32)
    sc = hip_ctx.scene_create(np.full(45, lod, np.int32), np.stack(w))
    oscene, _ = U.oracle_scene(oracle, [(v, t)], il, np.stack(w))
    rng = np.random.default_rng(4)
    n = 6000
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = rng.uniform(-1.0, -0.1, (n, 3))
    d = rng.uniform(0, 1e-6, (n, 3)) - rays[:, 0:3]
    d[n // 2:] += rng.uniform(0, 0.6, (n - n // 2, 3))
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 3] = S.MAX_SCENE_SIZE
    print("full stack", flush=True)
    gt, gi, gp, gb, st = hip_ctx.trace_closest(sc, rays)
    ot, oi, op, ob = oracle.trace_closest(oscene, rays)
    assert (st == 0).all() and (oi >= 0).sum() > 1000
    assert np.array_equal(gi, oi) and np.array_equal(gp, op)
    assert np.array_equal(gt.view(np.uint32), ot.view(np.uint32))
    assert np.array_equal(hip_ctx.trace_any(sc, rays), oracle.trace_any(oscene, rays))


@pytest.mark.parametrize("shift", [0.0, 0.3, 7.7])
@pytest.mark.parametrize("instances", [1, 2])
def test_coinciding_surfaces(hip_ctx, oracle, instances, shift):
    """Two sheets of different cells in one plane, and a fine one a few ulps
    beside them: at every ray two or three surfaces lie equally far to the last
    bits, their boxes are flat, and which of them is reported depends on the
    order of the leaves. Bit for bit the oracle's."""
    v, t = [], []
    for n, y in ((40, shift), (7, shift), (23, shift + 2e-7 * max(shift, 1.0))):
        gv, gt = _grid(n)
        t.append(gt + sum(len(x) for x in v))
        v.append(gv * np.float32([1.0, 0.0, 1.0]) + np.float32([0.013 * n, y, 0.007 * n]))
    v, t = np.concatenate(v).astype(np.float32), np.concatenate(t).astype(np.uint32)
    lod = hip_ctx.lod_create(v, t)
    hip_ctx.lbvh_build(lod)
    w = np.concatenate([S.IDENTITY34.reshape(1, 12), U.random_transforms(1, 5)])[:instances]
    il = np.zeros(instances, np.int32)
    sc = hip_ctx.scene_create(np.full(instances, lod, np.int32), w)
    oscene, _ = U.oracle_scene(oracle, [(v, t)], il, w)
    rng = np.random.default_rng(2)
    lo, hi = v.min(0), v.max(0)
    n = 100_000
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = lo + (hi - lo) * rng.random((n, 3)) + [0, 0.5, 0]
    rays[: n // 2, 1] += rng.random(n // 2) * 3
    d = rng.normal(size=(n, 3)) * [1, 0.3, 1] - [0, 1, 0]
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 3] = S.MAX_SCENE_SIZE
    print("coinciding surfaces, %d instances, shift %g" % (instances, shift), flush=True)
    gt, gi, gp, gb, st = hip_ctx.trace_closest(sc, rays)
    ot, oi, op, ob = oracle.trace_closest(oscene, rays)
    assert (oi >= 0).sum() > n // 5 and (st == 0).all()
    assert np.array_equal(gi, oi) and np.array_equal(gp, op)
    assert np.array_equal(gt.view(np.uint32), ot.view(np.uint32))
    hit = oi >= 0
    assert np.array_equal(gb[hit].view(np.uint32), ob[hit].view(np.uint32))
    assert np.array_equal(hip_ctx.trace_any(sc, rays), oracle.trace_any(oscene, rays))


@pytest.mark.parametrize("instances", [1, 40])
def test_persistent_queue_sizes(hip_ctx, oracle, instances):
    """Rays are handed to the lanes of persistent waves: fewer rays than a
    wave, rays that do not fill the waves (dealt out), and more than four
    chunks a wave (taken from the counter), with rays whose slab values are
    NaN (a zero direction component) among them, which take the reference
    traversal in the middle of a wave's work."""
    v, t = S.random_triangle_soup(3000, seed=6, mu=-3.0)
    w = np.concatenate([S.IDENTITY34.reshape(1, 12), U.random_transforms(instances - 1, 5)])[:instances]
    il = np.zeros(instances, np.int32)
    lod = hip_ctx.lod_create(v, t)
    hip_ctx.lbvh_build(lod)
    sc = hip_ctx.scene_create(np.full(instances, lod, np.int32), w)
    oscene, _ = U.oracle_scene(oracle, [(v, t)], il, w)
    rays = U.rays_toward(np.random.default_rng(1), 1_500_003, origin_box=(-1, 2), target_box=(0, 1))
    rays[::97, 4:7] = (0.0, 0.6, 0.8)
    print("persistent queue, %d instances" % instances, flush=True)
    full = hip_ctx.trace_closest(sc, rays)
    occ = hip_ctx.trace_any(sc, rays)
    m = 120_000
    ot, oi, op, _ = oracle.trace_closest(oscene, rays[:m])
    assert np.array_equal(full[2][:m], op) and np.array_equal(full[1][:m], oi)
    assert np.array_equal(full[0][:m].view(np.uint32), ot.view(np.uint32))
    assert np.array_equal(occ[:m], oracle.trace_any(oscene, rays[:m]))
    for n in (1, 7, 63, 65, 4099, 70_001, 400_003):
        got = hip_ctx.trace_closest(sc, rays[:n])
        assert all(np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b[:n]).view(np.uint32))
                   for a, b in zip(got, full)), n
        assert np.array_equal(hip_ctx.trace_any(sc, rays[:n]), occ[:n]), n
