"""Small passes, traced as whole paths by one kernel, against the queues'
kernels (a parking budget other than the default asks for them): the same
samples, the same sums in the same order, so the films are equal bit for bit,
and so are the ray counts."""
import pytest

import raycer_amd as ra
from raycer_amd import api
from tests.helpers import overlapping_scene

pytestmark = pytest.mark.gpu

SCENES = {
    "box": dict(kind=api.RCH_SCENE_BOX),
    "terrain": dict(kind=api.RCH_SCENE_TERRAIN, seed=1, grid=64),
    "soup": dict(kind=api.RCH_SCENE_SOUP, seed=3, tri_count=3000),
}


@pytest.fixture(scope="module")
def scenes(ctx):
    out = {}
    for name, kw in SCENES.items():
        kw = dict(kw)
        sd = ra.generate_scene(ra.scene_params(kw.pop("kind"), **kw))
        nodes, ordered, _, _ = ra.build_bvh(sd.vertices)
        out[name] = (sd, ctx.upload(sd, nodes, ordered))
    return out


# 2 x 2 pixels (lanes idle), odd sizes, one sample, one vertex, late and early
# roulette, exactly and just over what 256 compute units hold (262,144 paths)
@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("width,height,spp,length,rr,sampler", [
    (2, 2, 1, 1, 0, api.RC_SAMPLER_JITTERED),
    (61, 43, 1, 64, 3, api.RC_SAMPLER_CENTER),
    (67, 9, 4, 5, 0, api.RC_SAMPLER_CMJ),
    (256, 256, 4, 8, 1, api.RC_SAMPLER_RANDOM),
    (257, 255, 4, 3, 2, api.RC_SAMPLER_JITTERED),
])
def test_whole_paths_equal_the_queues(ctx, decision, scenes, name, width, height, spp, length, rr, sampler):
    sd, s = scenes[name]
    cfg = api.RenderCfg.from_buffer_copy(sd.desc.cfg)
    cfg.width, cfg.height, cfg.spp, cfg.max_path_length, cfg.rr_start, cfg.sampler = width, height, spp, length, rr, sampler
    film = ctx.film(width, height)
    results = []
    try:
        for tuning in (dict(park_steps=64), dict(), dict(stack_limit=1), dict(stack_limit=5)):
            ctx.set_tuning(**tuning)
            film.clear()
            ctx.render(s, film, sd.desc.camera, cfg)
            st = ctx.stats()
            results.append((film.sums().tobytes(), st.extension_rays, st.shadow_rays))
            assert st.parked_rays == 0 or "park_steps" in tuning
    finally:
        ctx.set_tuning()
        film.close()
    for r in results[1:]:
        assert r == results[0]


# At most as many paths as there are spill slots (2,048), but many more
# traversals that outgrow their rows than that: each claims a slot of its own,
# so paths are listed and walked again.  A frame of other samples comes first,
# so a path that is left out would show that frame's radiance.
@pytest.mark.parametrize("width,height", [(45, 45), (32, 64)])
@pytest.mark.parametrize("limit", [4, 5, 6, 7])
def test_small_passes_lose_no_listed_path(ctx, decision, width, height, limit):
    sd = overlapping_scene()
    nodes, ordered, _, _ = ra.build_bvh(sd.vertices)
    s = ctx.upload(sd, nodes, ordered)
    cfg = api.RenderCfg.from_buffer_copy(sd.desc.cfg)
    cfg.width, cfg.height, cfg.spp, cfg.max_path_length, cfg.rr_start = width, height, 1, 8, 0
    other = api.RenderCfg.from_buffer_copy(cfg)
    other.frame = cfg.frame + 5
    film = ctx.film(width, height)
    results = []
    try:
        for rows in (1, limit):
            ctx.set_tuning(stack_limit=1)
            ctx.render(s, film, sd.desc.camera, other)
            film.clear()
            ctx.set_tuning(stack_limit=rows)
            ctx.render(s, film, sd.desc.camera, cfg)
            st = ctx.stats()
            results.append((film.sums().tobytes(), st.extension_rays, st.shadow_rays))
    finally:
        ctx.set_tuning()
        film.close()
        s.close()
    assert results[1] == results[0]
    assert st.overflow_rays > 2048
