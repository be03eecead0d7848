"""The batched multi-scene form (rc_render_batch_tuned, rc_autotune_batch_plan)
on the 64-scene workload's own scenes.

The workload's soups (seed s: log-uniform 1k-500k triangles, 128^2-1024^2,
32 spp, depth 5) are rendered as one captured graph with autotuned plans and
concurrent branches; every film is checked against the FP64 oracle on seeded
pixels (same RNG keys, so the oracle replays the GPU's paths).  No seed of
0..63 draws both 400k+ triangles and 1024^2, so the set takes the largest
scene at 1024^2 (seed 23, 268,882 triangles), the largest overall (seed 33,
489,868 triangles at 128^2), the two other 400k-class scenes' resolutions
(seed 25: 409,165 at 512^2; seed 5: 367,448 at 256^2) and a ~1k-triangle
scene at each resolution.
"""
import numpy as np
import pytest

import oracle as orc
import raycer_amd as ra
from raycer_amd import api
from tests.conftest import ORACLE_THREADS

pytestmark = pytest.mark.gpu

SEEDS = [23, 33, 25, 5, 20, 1, 39, 28]


def load(ctx, seeds):
    out = []
    for seed in seeds:
        sd = ra.generate_scene(ra.scene_params(api.RCH_SCENE_SOUP, seed=seed))
        nodes, ordered, _, _ = ra.build_bvh(sd.vertices, method=api.RCH_BVH_BINNED)
        out.append((sd, ctx.upload(sd, nodes, ordered)))
    return out


def close(ctx, scenes, films):
    for f in films:
        f.close()
    for _, s in scenes:
        s.close()


def test_batch_workload_replays_the_oracle(ctx, tmp_path):
    scenes = load(ctx, SEEDS)
    sds = [sd for sd, _ in scenes]
    hs = [s for _, s in scenes]
    cams = [sd.desc.camera for sd in sds]
    cfgs = [sd.desc.cfg for sd in sds]
    assert {(c.width, c.spp, c.max_path_length) for c in cfgs} == {(w, 32, 5) for w in (128, 256, 512, 1024)}
    assert min(sd.ntri for sd in sds) < 1500 and max(sd.ntri for sd in sds) > 480000
    films = [ctx.film(c.width, c.height) for c in cfgs]
    try:
        plans, branches = ctx.autotune_batch_plan(hs, cams, cfgs, tmp_path / "tune.json")
        for p in plans:
            assert 1 <= p.spp_per_pass <= 32 and p.ext_block in (128, 256) and p.shadow_block in (64, 128, 256)
        assert branches in (1, 2, 4, 8)
        for f in films:
            f.clear()
        # two branches at least, so the concurrent form is the one checked
        ctx.render_batch_tuned(hs, films, cams, cfgs, plans, max(branches, 2))
        assert ctx.stats().samples == sum(c.width * c.height * c.spp for c in cfgs)
        rng = np.random.default_rng(11)
        for sd, cfg, film in zip(sds, cfgs, films):
            npix = cfg.width * cfg.height
            ids = np.sort(rng.choice(npix, 96, replace=False)).astype(np.uint32)
            ob = orc.BVH(sd.vertices)
            st = orc.render(ob, sd.tri_material, sd.materials, sd.desc.camera, orc.render_cfg(cfg, traversal=1),
                            pixel_ids=ids, threads=ORACLE_THREADS)
            sums = film.sums()[ids]
            np.testing.assert_allclose(sums[:, 3], st[:, 0], rtol=1e-5)  # film weights: the same samples
            gpu = film.linear()[ids, :3].astype(np.float64)
            ref = st[:, 2:5] / st[:, 0:1]
            equal = (np.abs(gpu - ref) <= 1e-4 * np.maximum(1.0, ref)).all(axis=1)
            print(f"soup {sd.ntri} tri {cfg.width}^2: {equal.mean():.1%} of sampled pixels replay the oracle")
            assert equal.mean() >= 0.95
            assert abs(gpu.mean() - ref.mean()) <= 0.02 * max(ref.mean(), 1e-3)
    finally:
        close(ctx, scenes, films)


def test_graph_relaunch_and_update(ctx):
    """The same batch relaunches the kept executable graph (no capture); a new
    frame index is captured again and the executable updated in place; each
    equals a fresh render of the scenes one by one."""
    scenes = load(ctx, [1, 28, 39])
    hs = [s for _, s in scenes]
    cams = [sd.desc.camera for sd, _ in scenes]
    cfgs = [sd.desc.cfg for sd, _ in scenes]
    for c in cfgs:
        c.width = c.height = 96
        c.spp = 4
    films = [ctx.film(c.width, c.height) for c in cfgs]
    plans = [api.BatchPlan(4, 256, 128, 0)] * len(hs)
    try:
        ctx.render_batch_tuned(hs, films, cams, cfgs, plans, 2)
        first = [f.sums() for f in films]
        assert ctx.stats().graph_relaunched == 0
        for f in films:
            f.clear()
        ctx.render_batch_tuned(hs, films, cams, cfgs, plans, 2)
        st = ctx.stats()
        assert st.graph_relaunched == 1 and st.graph_ms == 0.0
        assert all(f.sums().tobytes() == a.tobytes() for f, a in zip(films, first))
        for c in cfgs:
            c.frame = 9
        for f in films:
            f.clear()
        ctx.render_batch_tuned(hs, films, cams, cfgs, plans, 2)
        st = ctx.stats()
        assert st.graph_relaunched == 0 and st.graph_ms > 0.0
        ctx.set_tuning(spp_per_pass=4)
        try:
            for s, f, cam, cfg in zip(hs, films, cams, cfgs):
                f2 = ctx.film(cfg.width, cfg.height)
                ctx.render(s, f2, cam, cfg)
                assert f2.sums().tobytes() == f.sums().tobytes()
                f2.close()
        finally:
            ctx.set_tuning()
    finally:
        close(ctx, scenes, films)


def test_branches_and_block_shapes_do_not_change_the_images(ctx):
    """Block shapes change only the order of queue entries and the branches
    only which stream runs a frame; every slot's samples are keyed by pixel,
    sample and vertex, so the films are bit-identical to single renders."""
    scenes = load(ctx, [0, 2, 7, 9, 10])
    hs = [s for _, s in scenes]
    cams = [sd.desc.camera for sd, _ in scenes]
    cfgs = [sd.desc.cfg for sd, _ in scenes]
    for c in cfgs:
        c.width, c.height, c.spp = 80, 64, 4
    shapes = [(128, 64), (256, 256), (128, 128), (256, 64), (256, 128)]
    plans = [api.BatchPlan(2, e, s, 0) for e, s in shapes]
    films = [ctx.film(c.width, c.height) for c in cfgs]
    try:
        for br in (1, 3, 5):
            for f in films:
                f.clear()
            ctx.render_batch_tuned(hs, films, cams, cfgs, plans, br)
            got = [f.sums() for f in films]
            ctx.set_tuning(spp_per_pass=2)
            try:
                for i, (s, cam, cfg) in enumerate(zip(hs, cams, cfgs)):
                    f2 = ctx.film(cfg.width, cfg.height)
                    ctx.render(s, f2, cam, cfg)
                    assert f2.sums().tobytes() == got[i].tobytes(), (br, i)
                    f2.close()
            finally:
                ctx.set_tuning()
        with pytest.raises(ra.RaycerError):
            ctx.render_batch_tuned(hs, films, cams, cfgs, [api.BatchPlan(2, 96, 128, 0)] * 5, 1)
        with pytest.raises(ra.RaycerError):
            ctx.render_batch_tuned(hs, films, cams, cfgs, plans, 9)
    finally:
        close(ctx, scenes, films)


def test_plans_are_tuned_on_the_kernels_a_batch_runs(ctx, tmp_path):
    """Frames of several branches run the queues' kernels, whose block shapes a
    plan chooses; a small frame by itself is traced as whole paths, without a
    shadow launch.  The last frame the tuner times by itself tells which."""
    scenes = load(ctx, [1, 28])
    hs = [s for _, s in scenes]
    cams = [sd.desc.camera for sd, _ in scenes]
    cfgs = [sd.desc.cfg for sd, _ in scenes]
    for c in cfgs:
        c.width = c.height = 64
        c.spp = 4
    ctx.set_profiling(True)
    try:
        ctx.autotune_batch_plan(hs, cams, cfgs, tmp_path / "plan.json")
        assert ctx.stats().shadow_launches > 0
        ctx.autotune_batch(hs, cams, cfgs, tmp_path / "alone.json")  # one branch
        assert ctx.stats().shadow_launches == 0
    finally:
        ctx.set_profiling(False)
        close(ctx, scenes, [])
