"""Wavefront `rlpath` renderer on the GPU vs the CPU oracle.

At max depth 1 nothing learnt is used yet (the Q table and light CDFs are
read before their first update), so the film must equal the oracle's bit for
bit. Deeper, the Q proposals land through float atomics in a run-dependent
order, as in the reference, so the comparison is statistical: the GPU and the
oracle films must agree in mean and be equally close to a high-spp `path`
image of the same scene (rendered on the GPU, whose `path` films equal the
oracle's). In deterministic mode the table updates are summed per key in
sample order, the order in which the oracle adds them, so the films are equal
bit for bit at every depth and with rounds."""
import numpy as np
import pytest

import oracle
from cavalry_amd import render as R, scenes
from cavalry_amd.camera import for_scene

pytestmark = pytest.mark.gpu


def rel_mse(a, b):
    """mean over pixels and channels of (a - b)^2 / (b^2 + 1e-2)."""
    return float(np.mean((a - b) ** 2 / (b * b + 1e-2)))


@pytest.mark.parametrize("materials", ["matte", "mixed"])
def test_rlpath_depth1_matches_oracle_exactly(ctx, materials):
    print(f"[rlpath] depth 1 {materials}", flush=True)
    sc = scenes.cornell_box(seed=3, width=64, height=48, materials=materials)
    cam = for_scene(sc)
    rgb, w, rays = oracle.render_rlpath(sc, 4, cam, max_depth=1)
    scene = R.Scene(ctx, sc)
    film, st = R.render(ctx, scene, 4, integrator="rlpath", camera=cam, max_depth=1)
    np.testing.assert_array_equal(film.weight, w)
    same = float(np.mean(np.all(film.rgb.view(np.uint32) == rgb.view(np.uint32), axis=-1)))
    err = rel_mse(film.image, rgb / np.maximum(w, 1e-30)[..., None])
    print(f"[rlpath] identical pixels={same:.5f} rel_mse={err:.3e} rays={st['closest_rays'] + st['shadow_rays']} "
          f"oracle rays={rays}", flush=True)
    assert st["closest_rays"] + st["shadow_rays"] == rays
    assert same == 1.0
    scene.close()


@pytest.mark.parametrize("materials,depth", [("matte", 2), ("matte", 8), ("mixed", 8)])
def test_rlpath_statistically_matches_oracle(ctx, materials, depth):
    print(f"[rlpath] {materials} depth {depth}", flush=True)
    sc = scenes.cornell_box(seed=3, width=64, height=48, materials=materials)
    cam = for_scene(sc)
    scene = R.Scene(ctx, sc)
    ref_film, _ = R.render(ctx, scene, 1024, integrator="path", camera=cam, max_depth=depth)
    ref = ref_film.image
    spp = 16
    rgb, w, _ = oracle.render_rlpath(sc, spp, cam, max_depth=depth)
    ora = rgb / np.maximum(w, 1e-30)[..., None]
    film, st = R.render(ctx, scene, spp, integrator="rlpath", camera=cam, max_depth=depth)
    gpu = film.image
    e_gpu, e_ora = rel_mse(gpu, ref), rel_mse(ora, ref)
    m_gpu, m_ora, m_ref = float(gpu.mean()), float(ora.mean()), float(ref.mean())
    print(f"[rlpath] mean gpu={m_gpu:.5f} oracle={m_ora:.5f} path1024={m_ref:.5f} "
          f"rel_mse vs path1024: gpu={e_gpu:.3e} oracle={e_ora:.3e} gpu-vs-oracle={rel_mse(gpu, ora):.3e}",
          flush=True)
    assert np.isfinite(gpu).all()
    assert abs(m_gpu - m_ora) < 0.01 * m_ora
    assert abs(m_gpu - m_ref) < 0.02 * m_ref
    assert e_gpu < 1.25 * e_ora + 1e-5 and e_ora < 1.25 * e_gpu + 1e-5
    assert st["closest_rays"] > 0 and st["shadow_rays"] > 0
    scene.close()


def test_rlpath_grid_and_rate_options(ctx):
    sc = scenes.cornell_box(seed=4, width=48, height=48)
    cam = for_scene(sc)
    scene = R.Scene(ctx, sc)
    ref, _ = R.render(ctx, scene, 512, integrator="path", camera=cam)
    for grid, alpha in ((16, 1.0), (64, 0.3)):
        print(f"[rlpath] q_grid={grid} alpha_scale={alpha}", flush=True)
        film, _ = R.render(ctx, scene, 16, integrator="rlpath", camera=cam, q_grid=grid, alpha_scale=alpha)
        img = film.image
        assert np.isfinite(img).all()
        assert abs(float(img.mean()) - float(ref.image.mean())) < 0.03 * float(ref.image.mean())
    scene.close()


def test_rlpath_errors(ctx):
    from cavalry_amd._lib import CavError
    sc = scenes.cornell_box(width=8, height=8)
    scene = R.Scene(ctx, sc)
    with pytest.raises(CavError):
        R.render(ctx, scene, 1, integrator="rlpath", q_grid=65)
    with pytest.raises(CavError):
        R.render(ctx, scene, 1, integrator="rlpath", alpha_scale=1.5)
    with pytest.raises(CavError):
        R.render(ctx, scene, 1, integrator="rlpath", max_depth=80)  # 2 + 14 * 80 > 1024 dimensions
    with pytest.raises(ValueError):
        R.render(ctx, scene, 1, integrator="bdpt")
    scene.close()


def test_rlpath_rounds_match_oracle_rounds(ctx):
    """Learning carries over from round to round, on the GPU as in the oracle."""
    print("[rlpath] spp=8 in rounds of 2", flush=True)
    sc = scenes.cornell_box(seed=6, width=48, height=40)
    cam = for_scene(sc)
    rgb, w, _ = oracle.render_rlpath(sc, 8, cam, spp_per_round=2)
    ora = rgb / np.maximum(w, 1e-30)[..., None]
    scene = R.Scene(ctx, sc)
    film, st = R.render(ctx, scene, 8, integrator="rlpath", camera=cam, spp_per_round=2)
    assert st["rounds"] == 4
    np.testing.assert_array_equal(film.weight, w)
    err = rel_mse(film.image, ora)
    print(f"[rlpath] rounds: gpu-vs-oracle rel_mse={err:.3e} mean gpu={float(film.image.mean()):.5f} "
          f"oracle={float(ora.mean()):.5f}", flush=True)
    assert abs(float(film.image.mean()) - float(ora.mean())) < 0.01 * float(ora.mean())
    assert err < 1e-3
    scene.close()


@pytest.mark.parametrize("materials,kind", [("matte", "plain"), ("mixed", "plain"), ("metal", "sphere_light"),
                                            ("mixed", "rounds")])
def test_rlpath_deterministic_matches_oracle_exactly(ctx, materials, kind):
    """Deterministic table updates: the film equals the oracle's bit for bit
    at max depth 8 (learnt Q tables and light CDFs in use from the second
    bounce on), also across spp rounds, and two runs give the same film."""
    print(f"[rlpath] deterministic {materials} {kind}", flush=True)
    sc = scenes.cornell_box(seed=9, width=40, height=32, materials=materials,
                            lights="both" if kind == "sphere_light" else "quad")
    cam = for_scene(sc)
    spp, rnd = (8, 2) if kind == "rounds" else (4, 0)
    rgb, w, rays = oracle.render_rlpath(sc, spp, cam, max_depth=8, spp_per_round=rnd)
    scene = R.Scene(ctx, sc)
    film, st = R.render(ctx, scene, spp, integrator="rlpath", camera=cam, max_depth=8, spp_per_round=rnd,
                        deterministic=True)
    again, _ = R.render(ctx, scene, spp, integrator="rlpath", camera=cam, max_depth=8, spp_per_round=rnd,
                        deterministic=True)
    same = float(np.mean(np.all(film.rgb.view(np.uint32) == rgb.view(np.uint32), axis=-1)))
    print(f"[rlpath] identical pixels={same:.5f} rays={st['closest_rays'] + st['shadow_rays']} oracle={rays}",
          flush=True)
    np.testing.assert_array_equal(film.weight, w)
    np.testing.assert_array_equal(film.rgb, rgb)
    np.testing.assert_array_equal(again.rgb, film.rgb)
    assert st["closest_rays"] + st["shadow_rays"] == rays
    scene.close()


def test_rlpath_deterministic_after_buffers_grow(ctx):
    """A larger render in between reallocates the render buffers; the next
    deterministic render allocates its update records again and gives the
    same film as before (regression: its capacity was kept while the
    records were freed)."""
    print("[rlpath] deterministic, buffers grow in between", flush=True)
    sc = scenes.cornell_box(seed=5, width=32, height=24)
    big = scenes.cornell_box(seed=5, width=96, height=80)
    scene = R.Scene(ctx, sc)
    first, _ = R.render(ctx, scene, 2, integrator="rlpath", max_depth=4, deterministic=True)
    R.render(ctx, scene, 8, integrator="path", camera=for_scene(big), max_depth=2)
    again, _ = R.render(ctx, scene, 2, integrator="rlpath", max_depth=4, deterministic=True)
    np.testing.assert_array_equal(again.rgb, first.rgb)
    scene.close()


@pytest.mark.parametrize("nlights", [15, 16, 17, 64, 69])
def test_rlpath_light_counts(ctx, nlights):
    """The light statistics are finished a thread per entry below 16 lights and
    a wave per entry from there, 64 lights at a time: the deterministic film
    equals the oracle's bit for bit on both sides of each limit. (The scene's
    mirrors, glass and plastic take the bin masks of the Q distribution.)"""
    print(f"[rlpath] {nlights} lights", flush=True)
    sc = scenes.interior(0, seed=3, width=40, height=32, textures=False)
    lights = np.flatnonzero(sc.meshes["is_light"])
    assert len(lights) == 64
    sc.meshes["is_light"][lights[nlights:]] = 0
    sc.meshes["is_light"][:max(0, nlights - 64)] = 1  # (walls, above 64)
    sc.meshes["emission"][:max(0, nlights - 64)] = 1.5
    sc.meshes["emission"][sc.meshes["is_light"] == 0] = 0
    cam = for_scene(sc)
    rgb, w, rays = oracle.render_rlpath(sc, 4, cam, max_depth=6)
    scene = R.Scene(ctx, sc)
    film, st = R.render(ctx, scene, 4, integrator="rlpath", camera=cam, max_depth=6, deterministic=True)
    np.testing.assert_array_equal(film.weight, w)
    np.testing.assert_array_equal(film.rgb.view(np.uint32), rgb.view(np.uint32))
    assert st["closest_rays"] + st["shadow_rays"] == rays
    scene.close()
