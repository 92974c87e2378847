"""Traces over the wide tree vs the CPU oracle, bit for bit, at the sizes where
its build and its finishing pass can go wrong: trees of one node, of one
level, across the single-workgroup limit; rays that run along box planes,
coincident triangles, rays that hit nothing or come from very far, and more
undecided rays than the finishing pass's list holds."""
import numpy as np
import pytest

import oracle
from cavalry_amd import BVH, scenes, tune
from helpers import bits

pytestmark = pytest.mark.gpu


def _check(bvh, nd, tris, rays, lim, what):
    print(f"[wide] {what}: {len(tris)} triangles, {len(rays)} rays", flush=True)
    ref = oracle.trace_closest(nd, tris, rays)
    got = bvh.intersect(rays)
    np.testing.assert_array_equal(got["prim"], ref["prim"])
    for k in ("t", "u", "v"):
        np.testing.assert_array_equal(bits(got[k]), bits(ref[k]), err_msg=k)
    np.testing.assert_array_equal(bvh.test_visibility(rays, lim), oracle.trace_occluded(nd, tris, rays, lim))
    return ref


def _tree(ctx, tris, morton_bits, rounds):
    _, _, nd = oracle.lbvh_build(tris, morton_bits)
    if rounds:
        oracle.treelet_optimize(nd, rounds)
    return BVH.build(ctx, tris, optimization_rounds=rounds, morton_bits=morton_bits), nd


@pytest.mark.parametrize("n", [2, 3, 4, 5, 8, 9, 10, 31, 33, 257, 4096, 4097, 20000])
def test_sizes(ctx, n):
    rng = np.random.default_rng(n)
    tris = scenes.gmm_triangles(n, seed=n, edge=0.05 if n > 300 else 0.3)
    bvh, nd = _tree(ctx, tris, 30, 1 if n % 2 else 0)
    rays = scenes.random_rays(3000, seed=n + 1, lo=0.0, hi=1.0)
    lim = rng.uniform(0, 2, len(rays)).astype(np.float32)
    lim[::5] = np.inf
    _check(bvh, nd, tris, rays, lim, f"n={n}")


def _plane_rays(tris, n, seed):
    """Rays from points of the triangles (half exactly on them), most with one
    or two zero direction components of either sign."""
    rng = np.random.default_rng(seed)
    t = tris[rng.integers(0, len(tris), n)].reshape(n, 3, 3)
    b = rng.random((n, 2))
    s = np.sqrt(b[:, :1])
    p = (t[:, 0] * (1 - s) + t[:, 1] * (s * (1 - b[:, 1:])) + t[:, 2] * (s * b[:, 1:])).astype(np.float32)
    corner = rng.random(n) < 0.2
    p[corner] = t[corner, 1]
    d = rng.normal(size=(n, 3)).astype(np.float32)
    for share in (0.8, 0.2):
        k = np.nonzero(rng.random(n) < share)[0]
        d[k, rng.integers(0, 3, len(k))] = np.where(rng.random(len(k)) < 0.5, 0.0, -0.0)
    len_ = np.linalg.norm(d, axis=1, keepdims=True)
    d = np.where(len_ > 0, d / np.maximum(len_, 1e-20), d).astype(np.float32)
    o = np.where(rng.random((n, 1)) < 0.5, p, p + np.float32(1e-3) * d).astype(np.float32)
    return np.ascontiguousarray(np.concatenate([o, d], 1), np.float32)


@pytest.mark.parametrize("morton_bits,rounds", [(30, 0), (63, 3)])
def test_rays_along_planes_and_coincident_triangles(ctx, morton_bits, rounds):
    """The Cornell box (boxes standing on the floor, walls on the scene's own
    box planes) with some of its triangles doubled, one of them 70 times: rays
    along box planes, where the slab test meets 0 * inf, and equally near hits."""
    base = np.ascontiguousarray(scenes.cornell_box(seed=5).tris, np.float32)
    rng = np.random.default_rng(7)
    tris = np.concatenate([base, base[:40], base[rng.integers(0, len(base), 300)], np.repeat(base[2:3], 70, 0)])
    bvh, nd = _tree(ctx, tris, morton_bits, rounds)
    rays = _plane_rays(np.concatenate([base[:44], base[:44], tris[::37]]), 120000, 3)
    lim = rng.uniform(0, 2, len(rays)).astype(np.float32)
    lim[::5] = np.inf
    ref = _check(bvh, nd, tris, rays, lim, "planes")
    assert (ref["prim"] >= 0).sum() > 10000
    f = bvh.trace_fetches()
    assert f["long_closest_rays"] > 1000  # the finishing pass decided them


def test_odd_rays(ctx):
    """Rays outside what the wide tree's planes take: no direction, NaN,
    directions from 1e-38 to 1e30 long, origins beyond 2^40."""
    tris = scenes.gmm_triangles(3000, seed=3, edge=0.1)
    bvh, nd = _tree(ctx, tris, 30, 0)
    rays = scenes.random_rays(4000, seed=4, lo=0.0, hi=1.0)
    scale = np.float32([1e-30, 1e-20, 1e-6, 1e6, 1e20, 1e30])
    rays[:3000, 3:] *= scale[np.arange(3000) % 6][:, None]
    rays[3000:3100, 3:] = 0.0
    rays[3100:3200, 3] = np.nan
    rays[3200:3300, 0] = np.nan
    rays[3300:3400, 3:] *= np.float32(1e-38)
    rays[3400:3500, :3] -= rays[3400:3500, 3:] * np.float32(4e12)
    lim = np.full(len(rays), np.inf, np.float32)
    lim[::3] = 1.0
    lim[1::50] = np.nan
    _check(bvh, nd, tris, rays, lim, "odd")


def test_scene_far_from_the_origin_and_given_bounds(ctx):
    """Coordinates around 1e5 with small triangles, with scene bounds given
    that do not hold the triangles (the wide tree uses their own box)."""
    tris = (scenes.gmm_triangles(5000, seed=8, edge=0.05) + np.float32(1e5)).astype(np.float32)
    rays = scenes.random_rays(20000, seed=9, lo=0.0, hi=1.0)
    rays[:, :3] += np.float32(1e5)
    lim = np.full(len(rays), np.inf, np.float32)
    sb = np.float32([1e5 + 0.4] * 3 + [1e5 + 0.6] * 3)
    _, _, nd = oracle.lbvh_build(tris, 30, sb)
    bvh = BVH.build(ctx, tris, scene_bounds=sb)
    _check(bvh, nd, tris, rays, lim, "far")


def _reference_order(ctx, call):
    saved = tune.get_launch(ctx, tune.STANDALONE)
    try:
        tune.set_launch(ctx, tune.STANDALONE, dict(saved, handoff_steps=1 << 30))
        return call()
    finally:
        tune.set_launch(ctx, tune.STANDALONE, saved)


LIST = 1 << 20  # rays the finishing pass's list holds


def test_more_undecided_rays_than_the_list_holds(ctx):
    """Every triangle twice: every hit is undecided. More of them than the list
    holds; the rest are found by scanning. Compared with the reference's order
    on one lane per ray."""
    half = scenes.gmm_triangles(500, seed=11, edge=0.3)
    tris = np.ascontiguousarray(np.concatenate([half, half]), np.float32)
    n = LIST + 20011
    rays = scenes.random_rays(n, seed=12, lo=0.3, hi=0.7)
    bvh = BVH.build(ctx, tris)
    got = bvh.intersect(rays)
    f = bvh.trace_fetches()
    ref = _reference_order(ctx, lambda: bvh.intersect(rays))
    print(f"[wide] undecided: {f}, {(ref['prim'] >= 0).sum()} hits", flush=True)
    assert (ref["prim"] >= 0).sum() > LIST + 10000 and f["long_closest_rays"] == LIST  # (clamped to the list)
    np.testing.assert_array_equal(got["prim"], ref["prim"])
    for k in ("t", "u", "v"):
        np.testing.assert_array_equal(bits(got[k]), bits(ref[k]), err_msg=k)


def test_more_undecided_any_hit_rays_than_the_list_holds(ctx):
    """Walls standing on y = 0 and rays along that plane through their lower
    edges: every blocker is met along a plane of its box, where the sign of the
    direction's zero decides, so every ray is undecided."""
    rng = np.random.default_rng(22)
    x = np.arange(1, 41) / 41.0
    top = rng.uniform(0.2, 1, (40, 2))
    tris = np.stack([x, 0 * x, 0 * x, x, 0 * x, 0 * x + 1, x, top[:, 0], top[:, 1]], -1).astype(np.float32)
    n = LIST + 20011
    rays = np.zeros((n, 6), np.float32)
    rays[:, 0] = rng.uniform(-1, 0.9, n)
    rays[:, 2] = rng.uniform(0.05, 0.95, n)
    rays[:, 3] = 1.0
    rays[:, 4] = np.where(rng.random(n) < 0.5, 0.0, -0.0)
    lim = np.full(n, np.inf, np.float32)
    lim[::2] = 2.5
    bvh = BVH.build(ctx, tris)
    got = bvh.test_visibility(rays, lim)
    f = bvh.trace_fetches()
    ref = _reference_order(ctx, lambda: bvh.test_visibility(rays, lim))
    print(f"[wide] undecided any-hit: {f}, {int((ref == 0).sum())} blocked", flush=True)
    assert f["spilled_rays"] == LIST  # (clamped to the list)
    assert 0.2 < ref.mean() < 0.8
    np.testing.assert_array_equal(got, ref)
    few = slice(0, 5000)
    _, _, nd = oracle.lbvh_build(tris, 30)
    np.testing.assert_array_equal(got[few], oracle.trace_occluded(nd, tris, rays[few], lim[few]))


def test_rebuild_reuses_the_tree(ctx):
    """Rebuilds of one BVH object over other triangles, with and without
    rounds, leave no trace of the earlier tree."""
    import torch
    n = 30000
    bvh = None
    for k, rounds in enumerate((0, 3, 0)):
        tris = scenes.gmm_triangles(n, seed=40 + k, edge=0.01)
        dev = torch.from_numpy(tris).cuda()
        torch.cuda.synchronize()
        if bvh is None:
            bvh = BVH.build(ctx, dev, optimization_rounds=rounds, device=True)
        else:
            bvh.rebuild(dev, optimization_rounds=rounds)
        _, _, nd = oracle.lbvh_build(tris, 30)
        if rounds:
            oracle.treelet_optimize(nd, rounds)
        rays = scenes.random_rays(20000, seed=50 + k, lo=0.0, hi=1.0)
        lim = scenes.shadow_limits(len(rays), seed=60 + k)
        _check(bvh, nd, tris, rays, lim, f"rebuild {k}")


def _floor(k, size, axis=2, noise=0.0, seed=0):
    """k x k cells of two triangles each, side `size`, flat on `axis` but for
    noise of that size in its coordinate."""
    rng = np.random.default_rng(seed)
    g = np.linspace(0, size, k + 1)
    x, y = np.meshgrid(g, g, indexing="ij")
    p = np.stack([x, y, noise * rng.uniform(-1, 1, x.shape)], -1)
    a, b, c, d = p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]
    t = np.concatenate([np.stack(q, 2).reshape(-1, 3, 3) for q in ((a, b, c), (a, c, d))])
    return np.roll(t, axis - 2, axis=2)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("size", [2e-3, 1.0, 4000.0])
@pytest.mark.parametrize("noise", [0.0, 1e-17])
def test_rays_almost_along_flat_boxes(ctx, axis, size, noise):
    """Rays 1e-22 to 1e-9 of a floor's size above (below) it that sink to it
    (rise to it) over distances of its size: directions whose one component is
    far below the others, along boxes without extent on that axis. With noise,
    rays between the floor's lowest and highest vertex that do not move along
    its axis at all too."""
    rng = np.random.default_rng(int(axis + size) + (noise > 0))
    tris = np.ascontiguousarray(_floor(12, size, axis, noise * size).reshape(-1, 9), np.float32)
    n = 6000
    ang = rng.uniform(0, 2 * np.pi, n)
    h = size * 10.0 ** rng.uniform(-22, -9, n) * rng.choice([-1, 1], n)
    far = size * rng.uniform(0.05, 0.9, n)
    o = np.stack([*(rng.uniform(0, size, (2, n))), h], -1)
    d = np.stack([np.cos(ang), np.sin(ang), -h / far], -1)
    d[::3, 0] = 0.0
    if noise:
        o[::2, 2] = size * noise * rng.uniform(-0.9, 0.9, len(o[::2]))
        d[::2, 2] = rng.choice([0.0, -0.0], len(o[::2]))
    o, d = np.roll(o, axis - 2, 1), np.roll(d, axis - 2, 1)
    rays = np.ascontiguousarray(np.concatenate([o, d], 1), np.float32)
    lim = (size * rng.uniform(0, 2, n)).astype(np.float32)
    lim[::4] = np.inf
    bvh, nd = _tree(ctx, tris, 30, 0)
    ref = _check(bvh, nd, tris, rays, lim, f"axis {axis}, size {size}, noise {noise}")
    assert (ref["prim"] >= 0).sum() > 200


@pytest.mark.parametrize("size,length", [(1.0, 1e-38), (1.0, 2.4e-38), (1.0, 1e-36), (1e12, 1e-27), (1e10, 1e-30),
                                         (1e-13, 1.0), (1e-15, 1.0), (1e-7, 1e-14)])
def test_distances_near_the_limits_of_a_float(ctx, size, length):
    """Scenes and directions whose hits lie at distances up to infinity (the
    reference takes the first hit whatever its distance), and whose products
    in the triangle test lose bits to underflow."""
    tris = (scenes.gmm_triangles(700, seed=13, edge=0.4) * np.float32(size)).astype(np.float32)
    rays = scenes.random_rays(6000, seed=14, lo=0.2, hi=0.8)
    rays[:, :3] *= np.float32(size)
    rays[:, 3:] = (rays[:, 3:] * length).astype(np.float32)
    rays[::2, 4:] = 0.0
    lim = np.full(len(rays), np.inf, np.float32)
    lim[::3] = np.float32(size / length * 0.3) if size / length < 1e38 else np.float32(3e38)
    bvh, nd = _tree(ctx, tris, 30, 0)
    _check(bvh, nd, tris, rays, lim, f"size {size}, directions of {length}")


def _turned(tris, seed, size):
    q, _ = np.linalg.qr(np.random.default_rng(seed).normal(size=(3, 3)))
    return np.ascontiguousarray((tris @ q.T * size).reshape(-1, 9), np.float32), q


@pytest.mark.parametrize("size", [1.0, 10.0, 1e-3])
@pytest.mark.parametrize("walls", [False, True])
def test_rays_in_the_plane_of_a_turned_floor(ctx, size, walls):
    """Rays in the plane of a turned, tessellated floor meet its triangles edge
    on, where Moller-Trumbore's t is rounding noise that may lie far from the
    triangle's box; walls across the floor stop them at exact distances."""
    tris = _floor(40, 1.0)
    tris[..., :2] -= 0.5
    for x in (-0.2, 0.05, 0.3) if walls else ():
        w = tris[::7, :, [2, 1, 0]].copy()
        w[..., 0] = x
        tris = np.concatenate([tris, w])
    for seed in range(6):
        rng = np.random.default_rng(seed)
        tt, q = _turned(tris, seed, size)
        n = 8000
        o = np.stack([rng.uniform(-0.8, 0.8, n), rng.uniform(-0.8, 0.8, n), np.zeros(n)], -1)
        a = rng.uniform(0, 2 * np.pi, n)
        d = np.stack([np.cos(a), np.sin(a), rng.normal(size=n) * (0.0, 1e-8, 1e-7)[seed % 3]], -1)
        rays = np.ascontiguousarray(np.concatenate([o @ q.T * size, d @ q.T], 1), np.float32)
        bvh, nd = _tree(ctx, tt, 30, 3 * (seed % 2))
        ref, got = oracle.trace_closest(nd, tt, rays), bvh.intersect(rays)
        print(f"[wide] turned floor, size {size}, walls {walls}, seed {seed}: "
              f"{(ref['prim'] != got['prim']).sum()} of {n} differ; {bvh.trace_fetches()}", flush=True)
        np.testing.assert_array_equal(got["prim"], ref["prim"])
        for k in ("t", "u", "v"):
            np.testing.assert_array_equal(bits(got[k]), bits(ref[k]), err_msg=k)


@pytest.mark.parametrize("seed", [1323, 1394, 1432])
def test_determinants_that_round_to_zero(ctx, seed):
    """Rays in the plane of a coarse turned floor whose triangles before the
    nearest wall all have a determinant of exactly 0, the sum of terms that are
    not: one behind the wall rounds to something, and its t to less than the
    wall's."""
    rng = np.random.default_rng(seed)
    floor = _floor(int(rng.integers(3, 60)), 1.0)
    floor[..., :2] -= 0.5
    tris = [floor]
    for x in rng.uniform(-0.4, 0.4, rng.integers(0, 5)):
        all_ = np.concatenate(tris)
        w = all_[::int(rng.integers(1, 9)), :, [2, 1, 0]].copy()
        w[..., 0] = x
        tris = [np.concatenate([all_, w])]
    size = 10.0 ** rng.uniform(-3, 3)
    tt, q = _turned(tris[0], seed, size)
    shift = np.float32(0)
    if rng.random() < 0.3:
        shift = rng.uniform(-2, 2, 3).astype(np.float32)[np.tile([0, 1, 2], 3)] * np.float32(size)
    tt = (tt + shift).astype(np.float32)
    n = 60000
    o = np.stack([rng.uniform(-0.8, 0.8, n), rng.uniform(-0.8, 0.8, n), np.zeros(n)], -1)
    a = rng.uniform(0, 2 * np.pi, n)
    d = np.stack([np.cos(a), np.sin(a), rng.normal(size=n) * 10.0 ** rng.uniform(-9, -4) * (rng.random() < 0.7)], -1)
    at = tt.reshape(-1, 3).mean(0) - tris[0].reshape(-1, 3).mean(0) @ q.T * size
    rays = np.ascontiguousarray(np.concatenate([o @ q.T * size + at, d @ q.T], 1), np.float32)
    bvh, nd = _tree(ctx, tt, 30, int(rng.integers(0, 4)))
    ref, got = oracle.trace_closest(nd, tt, rays), bvh.intersect(rays)
    print(f"[wide] zero determinants, seed {seed}: {(ref['prim'] != got['prim']).sum()} differ", flush=True)
    np.testing.assert_array_equal(got["prim"], ref["prim"])
    np.testing.assert_array_equal(bits(got["t"]), bits(ref["t"]))


@pytest.mark.parametrize("ratio", [300, 30000, 3000000])
def test_needles(ctx, ratio):
    """Triangles `ratio` times longer than wide among ordinary ones, and rays
    aimed at them: edge on or not, their determinants are small."""
    rng = np.random.default_rng(ratio)
    base = scenes.gmm_triangles(3000, seed=15, edge=0.1)
    thin = scenes.gmm_triangles(3000, seed=16, edge=0.3).reshape(-1, 3, 3)
    thin[:, 2] = thin[:, 1] + (thin[:, 2] - thin[:, 1]) / np.float32(ratio)
    tris = np.ascontiguousarray(np.concatenate([base, thin.reshape(-1, 9)]), np.float32)
    n = 30000
    k, w = rng.integers(0, 3000, n), rng.random((n, 1))
    at = thin[k, 0] * (1 - w) + (thin[k, 1] + thin[k, 2]) / 2 * w
    o = rng.random((n, 3))
    d = at - o
    rays = np.ascontiguousarray(np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1), np.float32)
    # (with a limit, any-hit rays may skip a needle whose t lies far from its box: see cav_trace_launch)
    lim = np.full(n, np.inf, np.float32)
    bvh, nd = _tree(ctx, tris, 30, 0)
    _check(bvh, nd, tris, rays, lim, f"needles {ratio}")
    print(f"[wide] needles {ratio}: {bvh.trace_fetches()}", flush=True)


def test_which_tree_is_walked_and_what_it_cost(ctx):
    """trace_wide follows the launch shape and counts the triangles among the
    fetches; the build's stages (ms_wide among them) add up to its total."""
    tris = scenes.gmm_triangles(50000, seed=17, edge=0.01)
    bvh = BVH.build(ctx, tris, optimization_rounds=2)
    rays = scenes.random_rays(20000, seed=18, lo=0.0, hi=1.0)
    lim = scenes.shadow_limits(len(rays), seed=19)
    saved = tune.get_launch(ctx, tune.STANDALONE)
    try:
        for change, closest, occluded in (({}, True, True), ({"handoff_steps": 1 << 30}, False, False),
                                          ({"any_hit_step": 2}, True, False), ({"any_hit_whole_line": 1}, True, False)):
            tune.set_launch(ctx, tune.STANDALONE, dict(saved, **change))
            bvh.trace_fetches(reset=True)
            bvh.trace_wide(reset=True)
            bvh.intersect(rays)
            bvh.test_visibility(rays, lim)
            f, w = bvh.trace_fetches(), bvh.trace_wide()
            assert (w["closest"], w["occluded"]) == (closest, occluded), change
            for k in ("closest", "occluded"):
                assert (0 < w[k + "_triangles"] < f[k]) == w[k] and (w[k] or w[k + "_triangles"] == 0)
    finally:
        tune.set_launch(ctx, tune.STANDALONE, saved)
    st = bvh.stats()
    stages = sum(v for k, v in st.items() if k.startswith("ms_") and k != "ms_total")
    other = sum(ms for name, ms in bvh.kernel_times() if name in ("readback", "levels"))
    print(f"[wide] stages {stages:.4f} + {other:.4f} of {st['ms_total']:.4f} ms, wide {st['ms_wide']:.4f}", flush=True)
    assert st["ms_wide"] > 0 and abs(stages + other - st["ms_total"]) < 0.02 * st["ms_total"]


@pytest.mark.parametrize("n", [(1 << 21) - 3, 1 << 21, (1 << 21) + 1])
def test_build_in_the_place_of_the_records(ctx, n):
    """Above 2^21 triangles the wide tree is built where the traversal records
    go afterwards: its traces and the reference's (through those records) agree,
    also after a rebuild, and a build holds less memory per triangle."""
    import torch
    tris = scenes.gmm_triangles(n, seed=n & 255, edge=2e-3)
    dev = torch.from_numpy(tris).cuda()
    rays = scenes.random_rays(50000, seed=20, lo=0.0, hi=1.0)
    lim = scenes.shadow_limits(len(rays), seed=21)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    bvh = BVH.build(ctx, dev, device=True)
    held = (free - torch.cuda.mem_get_info()[0]) / n
    assert held < (500 if n <= 1 << 21 else 400)  # (371 and the allocations' rounding)
    saved = tune.get_launch(ctx, tune.STANDALONE)
    for again in (False, True):
        if again:
            bvh.rebuild(dev, optimization_rounds=1)
        got, vis = bvh.intersect(rays), bvh.test_visibility(rays, lim)
        try:
            tune.set_launch(ctx, tune.STANDALONE, dict(saved, handoff_steps=1 << 30))
            ref, rvis = bvh.intersect(rays), bvh.test_visibility(rays, lim)
        finally:
            tune.set_launch(ctx, tune.STANDALONE, saved)
        print(f"[wide] n={n}: {held:.0f} bytes a triangle, {(ref['prim'] >= 0).sum()} hits", flush=True)
        np.testing.assert_array_equal(got["prim"], ref["prim"])
        np.testing.assert_array_equal(bits(got["t"]), bits(ref["t"]))
        np.testing.assert_array_equal(vis, rvis)
    bvh.close()
