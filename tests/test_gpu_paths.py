"""Small passes, traced as whole paths by one kernel, against the queues'
kernels (a parking budget other than the default asks for them): the same
samples, the same sums in the same order, so the films are equal bit for bit,
and so are the ray counts."""
import pytest

import raycer_amd as ra
from raycer_amd import api

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
