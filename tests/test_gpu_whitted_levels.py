"""The Whitted tracer's offsets at the edges of their blocks: frames of 1 to a
few blocks of nodes (256) and of several rays per node, in one pass and cut
into passes of one sample per pixel.  The passes' trees are independent, so
both hold the same rays; only the grouping of the sums differs (one rounding
per pass of a pixel's sum: 1e-6 relative)."""
import numpy as np
import pytest

import raycer_amd as ra
from raycer_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(2, 2), (17, 15), (16, 16), (257, 1 + 1), (63, 129)])
@pytest.mark.parametrize("n", [0, 3])
def test_offsets_at_block_edges(ctx, width, height, n):
    sd = ra.generate_scene(ra.scene_params(api.RCH_SCENE_SPHERE_GROUND, seed=1, level=3, grid=16))
    nodes, ordered, _, _ = ra.build_bvh(sd.vertices)
    s = ctx.upload(sd, nodes, ordered)
    cfg = api.RenderCfg.from_buffer_copy(sd.desc.cfg)
    cfg.width, cfg.height, cfg.spp = width, height, 4
    L = sd.desc.light
    area = dict(area_light=1, area_n=n, area_radius=0.2) if n else {}
    lights = [api.light(api.RC_LIGHT_POINT, position=tuple(L.position), intensity=L.intensity,
                        max_distance=L.max_distance, attenuation=L.attenuation, **area)]
    settings = api.ray_settings(max_ray_iterations=2, ambient_intensity=0.1,
                                **(dict(ao_enabled=1, ao_n=n, ao_max_distance=0.3) if n else {}))
    mats = api.ray_materials(len(sd.materials), ray_reflectance=0.5, **(dict(refl_n=n, refl_glossiness=40.0) if n else {}))
    film = ctx.film(width, height)
    out = []
    try:
        for per_pass in (0, 1, 0):
            ctx.set_tuning(spp_per_pass=per_pass)
            film.clear()
            ctx.raytrace(s, film, sd.desc.camera, cfg, settings, mats, lights)
            out.append((film.linear(), ctx.stats().extension_rays, ctx.stats().shadow_rays))
    finally:
        ctx.set_tuning()
        film.close()
        s.close()
    assert out[0][1:] == out[1][1:]
    np.testing.assert_allclose(out[1][0], out[0][0], rtol=1e-6, atol=1e-7)
    assert out[2][0].tobytes() == out[0][0].tobytes()  # the order of the sums is fixed


# Levels of more than 1,024 blocks, which the scan's threads take several of:
# 1,033 blocks (most threads one, some two, the last none), 2,054 and 3,074.
# One sample per pass makes 259, 514 and 769, one to a thread.
@pytest.mark.parametrize("width,height", [(257, 257), (362, 363), (443, 444)])
@pytest.mark.parametrize("n", [0, 2])
def test_offsets_of_many_blocks(ctx, width, height, n):
    sd = ra.generate_scene(ra.scene_params(api.RCH_SCENE_SPHERE_GROUND, seed=1, level=3, grid=16))
    nodes, ordered, _, _ = ra.build_bvh(sd.vertices)
    s = ctx.upload(sd, nodes, ordered)
    cfg = api.RenderCfg.from_buffer_copy(sd.desc.cfg)
    cfg.width, cfg.height, cfg.spp = width, height, 4
    L = sd.desc.light
    area = dict(area_light=1, area_n=n, area_radius=0.2) if n else {}
    lights = [api.light(api.RC_LIGHT_POINT, position=tuple(L.position), intensity=L.intensity,
                        max_distance=L.max_distance, attenuation=L.attenuation, **area)]
    settings = api.ray_settings(max_ray_iterations=1, ambient_intensity=0.1,
                                **(dict(ao_enabled=1, ao_n=n, ao_max_distance=0.3) if n else {}))
    mats = api.ray_materials(len(sd.materials), ray_reflectance=0.5, **(dict(refl_n=n, refl_glossiness=40.0) if n else {}))
    film = ctx.film(width, height)
    out = []
    try:
        for per_pass in (1, 0):
            ctx.set_tuning(spp_per_pass=per_pass)
            film.clear()
            ctx.raytrace(s, film, sd.desc.camera, cfg, settings, mats, lights)
            out.append((film.linear(), ctx.stats().extension_rays, ctx.stats().shadow_rays))
    finally:
        ctx.set_tuning()
        film.close()
        s.close()
    assert out[1][1:] == out[0][1:]
    np.testing.assert_allclose(out[1][0], out[0][0], rtol=1e-6, atol=1e-7)
