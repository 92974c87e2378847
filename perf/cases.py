"""The work a user of this framework has it do, as cases that can be timed.

Five kinds of call, each through the public entry points:

  frame   a moving scene: rebuild the BVH of device-resident triangles (LBVH and
          0 to 10 treelet rounds, 30- or 63-bit Morton codes), then trace the
          frame's rays (closest hits with barycentrics; half of the cases also
          shadow rays). What the benchmark's step does.
  trace   rays over a resident BVH: primary rays of a camera, diffuse bounce
          rays from the surfaces, or shadow rays towards the lights that ignore
          their source and target meshes.
  query   host-side queries (picking, collision): numpy rays in, numpy hits and
          visibility out, over a small or medium scene.
  render  whole films: path, rlpath and directlighting on the Cornell box
          (Halton, 512^2 x 16 and smaller) and on textured procedural interiors.
  serve   a render server with resident scenes: a burst of small mixed requests,
          submitted together and polled until their films are ready.

Ranges: 2000 to 2^22 triangles, 1000 to 2^21 rays, films of 64 x 36 to
1920 x 1080 pixels and 1 to 16 samples per pixel, depth 2 to 16. Sizes follow
the repository's benchmark (Cornell box 512^2 x 16 at depth 8, interiors of 0.1M
to 2M triangles at depth 16, Gaussian-mixture soups) and its tests.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cavalry_amd import BVH, Context, render as R, scenes
from cavalry_amd._lib import check, lib
from cavalry_amd.camera import look_at
from cavalry_amd.serve import Server

DEV = "cuda:0"
_CTX = None


def _ctx() -> Context:
    """The program's one context (device and stream)."""
    global _CTX
    if _CTX is None:
        _CTX = Context(0)
    return _CTX


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: a toy scene rebuilt and traced each frame; launches and host work count
        dict(name="frame_3k", kind="frame", geo="soup", n=3001, bits=30, rounds=0, rays="bounce", nrays=4096, shadow=True),
        # a moving scene of ordinary size, rebuilt each frame without treelet rounds
        dict(name="frame_1M", kind="frame", geo="interior", n=1_000_000, bits=30, rounds=0, rays="camera", nrays=131_072, shadow=False),
        # scene load: the front end's 63-bit codes and the default 3 treelet rounds at a large, odd size
        dict(name="frame_4M_r3", kind="frame", geo="soup", n=3_999_971, bits=63, rounds=3, rays="bounce", nrays=30_001, shadow=False),
        # the benchmark's step (build, 3 rounds, random closest-hit and shadow rays) at a quarter million rays
        dict(name="step_1M", kind="frame", geo="soup", n=1 << 20, bits=30, rounds=3, rays="random", nrays=1 << 18, shadow=True),
        # primary rays of a full-HD view: coherent
        dict(name="camera_1M", kind="trace", geo="interior", n=1_000_000, rounds=3, rays="camera", nrays=2_073_600),
        # diffuse bounce rays: incoherent
        dict(name="bounce_1M", kind="trace", geo="interior", n=1_000_000, rounds=3, rays="bounce", nrays=1_048_573),
        # next-event rays from the surfaces to the lights, their meshes ignored
        dict(name="shadow_1M", kind="trace", geo="interior", n=1_000_000, rounds=3, rays="shadow", nrays=2_073_600),
        # picking / collision queries from host arrays
        dict(name="query_200k", kind="query", geo="soup", n=200_000, rounds=3, nrays=50_001),
        # the benchmark's Cornell-box render
        dict(name="path_cornell", kind="render", scene="cornell", n=0, integrator="path", width=512, height=512, spp=16,
             depth=8, rounds=0, q_grid=32, det=False, sort=False),
        # path tracing at scale: a textured interior, deep paths
        dict(name="path_interior", kind="render", scene="interior", n=1_000_000, integrator="path", width=1280, height=720,
             spp=8, depth=16, rounds=3, q_grid=32, det=False, sort=False),
        # guided path tracing on an interior: the Q table's work, its updates by float atomics (the default), hits sorted
        dict(name="rlpath_interior", kind="render", scene="interior", n=400_000, integrator="rlpath", width=480, height=270,
             spp=16, depth=8, rounds=3, q_grid=32, det=False, sort=True),
        # a burst of small requests on two resident scenes
        dict(name="serve_burst", kind="serve", n=100_000, requests=12, width=256, height=144, spp=4, depth=8, graphs=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "trace", "trace", "query", "render", "render", "serve"])
    if kind == "frame":
        n = _log_int(rng, 2000, 3_000_000)
        rays = rng.choice(["bounce", "random"] if n < 300_000 else ["bounce"])
        return dict(kind=kind, geo="soup", n=n, bits=rng.choice([30, 63]), rounds=rng.choice([0, 0, 1, 3, 10] if n < 1_000_000 else [0, 1, 3]),
                    rays=rays, nrays=_log_int(rng, 1000, 200_000), shadow=rng.random() < 0.5)
    if kind == "trace":
        return dict(kind=kind, geo=rng.choice(["interior", "soup"]), n=_log_int(rng, 100_000, 1_000_000), rounds=rng.choice([0, 3]),
                    rays=rng.choice(["camera", "bounce", "shadow"]), nrays=_log_int(rng, 1000, 2_000_000))
    if kind == "query":
        return dict(kind=kind, geo="soup", n=_log_int(rng, 2000, 400_000), rounds=rng.choice([0, 3]), nrays=_log_int(rng, 1000, 100_000))
    if kind == "render":
        integrator = rng.choice(["path", "path", "rlpath", "directlighting"])
        scene = rng.choice(["cornell", "cornell_mixed", "interior"])
        w = _log_int(rng, 64, 960)
        return dict(kind=kind, scene=scene, n=_log_int(rng, 100_000, 500_000) if scene == "interior" else 0, integrator=integrator,
                    width=w, height=max(1, w * 9 // 16), spp=_log_int(rng, 1, 16), depth=rng.randint(2, 8),
                    rounds=rng.choice([0, 3]), q_grid=rng.choice([16, 32]), det=integrator == "rlpath" and rng.random() < 0.6,
                    sort=rng.random() < 0.4)
    return dict(kind=kind, n=_log_int(rng, 100_000, 200_000), requests=rng.randint(3, 16), width=_log_int(rng, 64, 320), height=rng.randint(64, 180),
                spp=rng.randint(1, 6), depth=rng.randint(3, 8), graphs=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _unit(g, n):
    v = torch.randn(n, 3, generator=g, device=DEV)
    return v / v.norm(dim=1, keepdim=True).clamp_min(1e-20)


def _soup(n, seed, edge=1e-3, components=8):
    """The benchmark's Gaussian-mixture soup: clustered small triangles in the
    unit cube, log-normal vertex offsets (median `edge`), random orientation."""
    g = _gen(seed)
    means = 0.15 + 0.7 * torch.rand(components, 3, generator=g, device=DEV)
    sig = 0.03 + 0.09 * torch.rand(components, generator=g, device=DEV)
    comp = torch.randint(components, (n,), generator=g, device=DEV)
    c = (means[comp] + torch.randn(n, 3, generator=g, device=DEV) * sig[comp, None]).clamp(0, 1)
    v = [c + torch.exp(math.log(edge) + 0.7 * torch.randn(n, 1, generator=g, device=DEV)) * _unit(g, n) for _ in range(3)]
    return torch.cat(v, 1).contiguous()


def _interior(n, seed, width=64, height=36, depth=8):
    return scenes.interior(n, seed=1 + seed % 1000, width=width, height=height, max_depth=depth, tex_size=256)


def _surface_points(tris, g, n):
    """Uniform points on n random triangles and their unit normals."""
    t = tris[torch.randint(len(tris), (n,), generator=g, device=DEV)].view(n, 3, 3)
    b = torch.rand(n, 2, generator=g, device=DEV)
    s = b[:, :1].sqrt()
    p = t[:, 0] * (1 - s) + t[:, 1] * (s * (1 - b[:, 1:])) + t[:, 2] * (s * b[:, 1:])
    m = torch.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0], dim=1)
    return p, m / m.norm(dim=1, keepdim=True).clamp_min(1e-20)


def _camera_rays(lo, hi, g, n):
    """Jittered pinhole rays, row by row over a 16:9 film, from near the front
    of the scene's box into it."""
    w = max(1, round(math.sqrt(n * 16 / 9)))
    i = torch.arange(n, device=DEV)
    rows = (n + w - 1) // w
    x = ((i % w).float() + torch.rand(n, generator=g, device=DEV)) / w - 0.5
    y = 0.5 - ((i // w).float() + torch.rand(n, generator=g, device=DEV)) / rows
    eye = lo + (hi - lo) * torch.tensor([0.5, 0.5, 0.03], device=DEV)
    d = torch.stack([x * 1.78, y, torch.full_like(x, 0.87)], 1)
    d = d / d.norm(dim=1, keepdim=True)
    return torch.cat([eye.expand(n, 3), d], 1).contiguous()


def _bounce_rays(tris, g, n):
    """Cosine-distributed rays from the surfaces, started 1e-3 along the ray."""
    p, m = _surface_points(tris, g, n)
    d = m * torch.where(torch.rand(n, 1, generator=g, device=DEV) < 0.5, 1.0, -1.0) + 0.999 * _unit(g, n)
    d = d / d.norm(dim=1, keepdim=True)
    return torch.cat([p + 1e-3 * d, d], 1).contiguous()


def _random_rays(g, n):
    """The benchmark's rays: origins uniform in [-0.5, 1.5]^3, any direction."""
    return torch.cat([2 * torch.rand(n, 3, generator=g, device=DEV) - 0.5, _unit(g, n)], 1).contiguous()


def _lo_hi(tris):
    v = tris.view(-1, 3)
    return v.amin(0), v.amax(0)


def _rays(kind, tris, g, n):
    if kind == "camera":
        return _camera_rays(*_lo_hi(tris), g, n)
    if kind == "random":
        return _random_rays(g, n)
    return _bounce_rays(tris, g, n)


def _shadow_rays(tris, mesh, g, n):
    """From surface points to points on other triangles (an interior's last
    meshes before the objects are its lights; any target costs the same), with
    the target's distance as limit and both meshes ignored."""
    i, j = (torch.randint(len(tris), (n,), generator=g, device=DEV) for _ in range(2))
    lights = (mesh >= 6) & (mesh < 70)  # the interior's ceiling lights
    if bool(lights.any()):
        ids = lights.nonzero()[:, 0]
        j = ids[j % len(ids)]
    p, q = (tris[k].view(n, 3, 3).mean(1) for k in (i, j))
    d = q - p
    lim = d.norm(dim=1).clamp_min(1e-6)
    return (torch.cat([p, d / lim[:, None]], 1).contiguous(), lim.contiguous(), mesh[i].contiguous(), mesh[j].contiguous())


def _geometry(case, seed):
    """Triangles [n, 9] and mesh ids on the GPU."""
    if case["geo"] == "interior":
        a = _interior(case["n"], seed)
        return (torch.from_numpy(a.tris).to(DEV), torch.from_numpy(a.tri_mesh).to(DEV))
    t = _soup(case["n"], seed)
    return t, (torch.arange(len(t), device=DEV, dtype=torch.int32) * 64 // len(t)).to(torch.int32)


def _closest_out(n):
    return dict(prim=torch.empty(n, dtype=torch.int32, device=DEV), **{k: torch.empty(n, device=DEV) for k in "tuv"})


def _prepare_rays(case, seed):
    ctx = _ctx()
    tris, mesh = _geometry(case, seed)
    g = _gen(seed + 7919)
    n = case["nrays"]
    s = dict(case=case, ctx=ctx, tris=tris)
    if case["rays"] != "shadow":
        s["rays"], s["hits"] = _rays(case["rays"], tris, g, n), _closest_out(n)
    if case["rays"] == "shadow" or case.get("shadow"):
        s["srays"], s["lim"], s["src"], s["dst"] = _shadow_rays(tris, mesh, g, n)
        s["vis"] = torch.empty(n, dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    s["bvh"] = BVH.build(ctx, tris, optimization_rounds=case["rounds"], morton_bits=case.get("bits", 30), tri_mesh=mesh, device=True)
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("frame", "trace"):
        return _prepare_rays(case, seed)
    ctx = _ctx()
    if kind == "query":
        tris = _soup(case["n"], seed, edge=5e-3)
        g = _gen(seed + 7919)
        rays, srays = _bounce_rays(tris, g, case["nrays"]), _random_rays(g, case["nrays"])
        lim = 2 * math.sqrt(3) * torch.rand(case["nrays"], generator=g, device=DEV)
        h = [v.cpu().numpy() for v in (tris, rays, srays, lim)]
        return dict(case=case, bvh=BVH.build(ctx, h[0], optimization_rounds=case["rounds"]), rays=h[1], srays=h[2], lim=h[3])
    if kind == "render":
        a = _render_arrays(case, seed)
        scene = R.Scene(ctx, a, bvh_rounds=case["rounds"])
        return dict(case=case, ctx=ctx, scene=scene, camera=_view(a, seed, case["width"], case["height"]))
    # serve (the server first: it is closed before the scenes that it holds)
    arrays = [_interior(case["n"], seed, depth=case["depth"]), scenes.cornell_box(seed=1 + seed % 1000, materials="mixed", max_depth=case["depth"])]
    server = Server(ctx, arena_bytes=4 << 30, host_arena_bytes=64 << 20, pool_tasks=1 << 20, use_graphs=case["graphs"])
    sc = [R.Scene(ctx, a, bvh_rounds=3) for a in arrays]
    reqs = []
    for k in range(case["requests"]):  # half path, a quarter each rlpath and directlighting; sizes vary
        w, h = max(16, case["width"] >> (k % 3)), max(16, case["height"] >> (k % 3))
        reqs.append((k % 2, _view(arrays[k % 2], seed + k, w, h), ("path", "rlpath", "path", "directlighting")[k // 2 % 4]))
    return dict(case=case, server=server, scenes=sc, requests=reqs)


def _render_arrays(case, seed):
    if case["scene"] == "interior":
        return _interior(case["n"], seed, case["width"], case["height"], case["depth"])
    mixed = case["scene"] == "cornell_mixed"
    return scenes.cornell_box(seed=1 + seed % 1000, width=case["width"], height=case["height"], max_depth=case["depth"],
                              materials="mixed" if mixed else "matte", smooth=mixed, textured=mixed, env=mixed)


def _view(a, seed, width, height):
    """The scene's camera, its eye moved a little by the seed."""
    j = np.random.default_rng(seed).uniform(-0.1, 0.1, 3).astype(np.float32)
    return look_at(a.eye + j, a.center, a.up, a.fov, width, height)


# ------------------------------------------------------------------ one pass
def _ptr(t):
    return None if t is None else t.data_ptr()


def _closest(s):
    o = s["hits"]
    check(s["ctx"].handle, lib().cav_trace_closest_device(
        s["ctx"].handle, s["bvh"].handle, _ptr(s["rays"]), len(s["rays"]), _ptr(o["prim"]), _ptr(o["t"]), _ptr(o["u"]), _ptr(o["v"])))
    return o


def _occluded(s):
    check(s["ctx"].handle, lib().cav_trace_occluded_device(
        s["ctx"].handle, s["bvh"].handle, _ptr(s["srays"]), _ptr(s["lim"]), _ptr(s["src"]), _ptr(s["dst"]), len(s["srays"]), _ptr(s["vis"])))
    return s["vis"]


def run(state):
    c = state["case"]
    if c["kind"] in ("frame", "trace"):
        if c["kind"] == "frame":
            state["bvh"].rebuild(state["tris"], optimization_rounds=c["rounds"], morton_bits=c["bits"])
        out = {}
        if "rays" in state:
            out.update(_closest(state))
        if "srays" in state:
            out["visible"] = _occluded(state)
        return out
    if c["kind"] == "query":
        out = state["bvh"].intersect(state["rays"])
        out["visible"] = state["bvh"].test_visibility(state["srays"], state["lim"])
        return out
    if c["kind"] == "render":
        film, _ = R.render(state["ctx"], state["scene"], c["spp"], integrator=c["integrator"], camera=state["camera"], max_depth=c["depth"],
                           q_grid=c["q_grid"], sort_by_material=c["sort"], deterministic=c["det"])
        return dict(rgb=film.rgb, weight=film.weight)
    srv = state["server"]
    tickets = [srv.submit(state["scenes"][k], c["spp"], integrator=integ, camera=cam, max_depth=c["depth"], q_grid=16, deterministic=True)
               for k, cam, integ in state["requests"]]
    out = {}
    for i, t in enumerate(tickets):
        assert srv.poll(t)["status"] == 2  # CAV_SERVE_DONE
        out["rgb%02d" % i], out["weight%02d" % i] = t.film.rgb, t.film.weight
    return out


# ------------------------------------------------------------------ work, tolerance, reference
# a ray over a balanced tree: two box tests per level (about 24 operations each) and two triangle tests (about 40)
def _ray_flops(n):
    return 48 * math.log2(max(n, 2)) + 80


def work(case):
    """Each input read once and each output written once; operations of the
    box and triangle tests that a balanced tree needs, and of the shading."""
    kind = case["kind"]
    if kind in ("frame", "trace", "query"):
        n, r = case["n"], case["nrays"]
        both = kind == "query" or case.get("shadow")
        closest = 0 if case["rays" if kind != "query" else "kind"] == "shadow" else 1
        b = 36 * n + closest * r * 40 + (r * 37 if both or not closest else 0)
        f = (closest + (1 if both or not closest else 0)) * r * _ray_flops(n)
        if kind == "frame":  # the tree's 2n - 1 boxes; one combined box per inner node, 119 subset costs per 7-leaf treelet
            b += 64 * n
            f += 30 * n + case["rounds"] * n / 3 * 2000
        return {"bytes": b, "flops": f}
    if kind == "render":
        px, n = case["width"] * case["height"], max(case["n"], 4014)
        depth = 1 if case["integrator"] == "directlighting" else min(case["depth"], 4)
        per = 2 * _ray_flops(n) + 400 + (128 * 60 if case["integrator"] == "rlpath" else 0)
        return {"bytes": 16 * px + 36 * n, "flops": px * case["spp"] * depth * per}
    px = sum((max(16, case["width"] >> (k % 3)) * max(16, case["height"] >> (k % 3))) for k in range(case["requests"]))
    return {"bytes": 16 * px + 36 * (case["n"] + 4014), "flops": px * case["spp"] * min(case["depth"], 4) * (2 * _ray_flops(case["n"]) + 400)}


def tolerance(case):
    """Hits, visibility and films are reproducible bit for bit: every float
    expression is evaluated in one written order, sums have one fixed order.
    Not so rlpath with its default float-atomic table updates, whose order
    varies: two films of one input differ by up to 3.3e-5 (2-norm) and 0.0092
    (largest, against the film's root mean square) at depth 8 on the interior
    and by 1.1e-6 and 1.8e-4 on the Cornell boxes; four times that here."""
    if case["kind"] == "render" and case["integrator"] == "rlpath" and not case["det"]:
        return {"rel": 1.4e-4, "max": 0.04}
    return "exact"


def exact(case, seed):
    """Closest hits by testing every triangle in binary64 (hit distance and
    barycentrics; ids and visibility are whole values)."""
    kind = case["kind"]
    if kind not in ("frame", "trace", "query") or (kind == "trace" and case["rays"] == "shadow") or case["n"] * case["nrays"] > 2.5e10:
        return None
    if kind == "query":
        tris, g = _soup(case["n"], seed, edge=5e-3), _gen(seed + 7919)
        rays = _bounce_rays(tris, g, case["nrays"])
    else:
        tris, _ = _geometry(case, seed)
        rays = _rays(case["rays"], tris, _gen(seed + 7919), case["nrays"])
    v = tris.double()
    v0, e1, e2 = v[:, :3], v[:, 3:6] - v[:, :3], v[:, 6:] - v[:, :3]
    out = {k: [] for k in "tuv"}
    step = max(1, (1 << 24) // len(v))
    cross = lambda a, b: (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])
    dot = lambda a, b: a[0] * b[0] + a[1] * b[1] + a[2] * b[2]
    cols = lambda m: tuple(m[:, k][None, :] for k in range(3))
    V0, E1, E2 = cols(v0), cols(e1), cols(e2)
    for at in range(0, len(rays), step):
        r = rays[at:at + step].double()
        o, d = (tuple(r[:, k + s][:, None] for k in range(3)) for s in (0, 3))
        tv = tuple(o[k] - V0[k] for k in range(3))
        pv = cross(d, E2)
        inv = 1 / dot(E1, pv)
        u = dot(tv, pv) * inv
        qv = cross(tv, E1)
        w = dot(d, qv) * inv
        t = dot(E2, qv) * inv
        ok = (u >= 0) & (u <= 1) & (w >= 0) & (u + w <= 1) & (t > 0) & torch.isfinite(inv)
        t = torch.where(ok, t, math.inf)
        best, i = t.min(1)
        hit = torch.isfinite(best)
        for k, x in (("t", best), ("u", u.gather(1, i[:, None])[:, 0]), ("v", w.gather(1, i[:, None])[:, 0])):
            out[k].append(torch.where(hit, x, torch.zeros_like(x)))
    got = {k: torch.cat(x) for k, x in out.items()}
    if kind == "query":
        got = {k: x.cpu().numpy() for k, x in got.items()}
    return dict(got, prim=None, **({"visible": None} if kind == "query" or case.get("shadow") else {}))
