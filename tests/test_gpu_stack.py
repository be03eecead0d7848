"""Traversal stacks that outgrow their on-chip rows.

A lane whose rows are full moves them to a spill slot in global memory and
goes on; when the launch's slots (2048, or one for 16 rays) are taken the ray is walked again by the
deep-stack kernel.  A limit below four rows spills nothing, so one row sends
every ray that needs more to the deep-stack kernel: the general path, against
which the others are compared bit for bit (the hit does not depend on where a
stack is kept).
"""
import numpy as np
import pytest

import raycer_amd as ra
from raycer_amd import api
from tests.helpers import random_rays

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def soup(ctx):
    sd = ra.generate_scene(ra.scene_params(api.RCH_SCENE_SOUP, seed=11, tri_count=40000))
    nodes, ordered, _, _ = ra.build_bvh(sd.vertices)
    return sd, ctx.upload(sd, nodes, ordered)


def query_rays(sd, n):
    v = sd.vertices.reshape(-1, 3)
    rays = random_rays(n, 5, v.min(0), v.max(0))
    f = rays.view(np.float32).reshape(-1, 8)
    f[1::4, 4:7] = np.eye(3, dtype=np.float32)[np.arange(len(f[1::4])) % 3]  # along the axes
    f[2::4, 3], f[2::4, 7] = 0.05, 0.8  # a finite range
    return rays


@pytest.mark.parametrize("limit", [3, 4, 5, 7, 19, 0])
@pytest.mark.parametrize("n", [1, 65, 2048, 2049, 60000])
def test_spilled_stacks_give_the_same_hits(ctx, decision, soup, n, limit):
    sd, s = soup
    rays = query_rays(sd, n)
    results = []
    try:
        for rows in (1, limit):
            ctx.set_tuning(stack_limit=rows)
            hits = ctx.trace_closest(s, rays)
            outgrown = ctx.stats().overflow_rays
            occ = ctx.trace_any(s, rays)
            assert ctx.stats().overflow_rays <= n
            results.append((hits.tobytes(), np.asarray(occ).tobytes(), outgrown))
    finally:
        ctx.set_tuning()
    (h0, o0, all_rays), (h1, o1, outgrown) = results
    assert h1 == h0 and o1 == o0
    print(f"{n} rays, {limit} rows: {outgrown} outgrew them ({all_rays} one row)")
    assert outgrown <= all_rays
    if n == 60000 and limit in (3, 4):
        assert outgrown > n // 16  # more than there are slots: both ways are taken


# As many slots as a traversal's word can name (131,071), and fewer.
@pytest.mark.parametrize("n", [600_001, 2_200_000])
@pytest.mark.parametrize("limit", [4, 5])
def test_many_slots(ctx, decision, soup, n, limit):
    sd, s = soup
    rays = query_rays(sd, n)
    results = []
    try:
        for rows in (0, limit):
            ctx.set_tuning(stack_limit=rows)
            hits = ctx.trace_closest(s, rays)
            outgrown = ctx.stats().overflow_rays
            results.append((hits.tobytes(), np.asarray(ctx.trace_any(s, rays)).tobytes()))
    finally:
        ctx.set_tuning()
    assert results[1] == results[0]
    assert outgrown > min(n // 16, 131071)


@pytest.mark.parametrize("limit", [4, 6])
def test_spilled_and_parked_traversals_give_the_same_image(ctx, decision, soup, limit):
    """A parked traversal keeps its spill slot over the resume kernels."""
    sd, s = soup
    cfg = api.RenderCfg.from_buffer_copy(sd.desc.cfg)
    cfg.width, cfg.height, cfg.spp, cfg.max_path_length = 61, 47, 4, 4
    film = ctx.film(cfg.width, cfg.height)
    sums = []
    try:
        for tuning in (dict(stack_limit=1, park_steps=0), dict(stack_limit=limit, park_steps=0),
                       dict(stack_limit=limit, park_steps=4)):
            ctx.set_tuning(**tuning)
            film.clear()
            ctx.render(s, film, sd.desc.camera, cfg)
            sums.append(film.sums().tobytes())
            assert ctx.stats().overflow_rays > 0
        assert ctx.stats().parked_rays > 0
    finally:
        ctx.set_tuning()
        film.close()
    assert sums[1] == sums[0] and sums[2] == sums[0]


@pytest.mark.parametrize("ntri", [3, 10, 50, 100])
def test_unused_slots_seen_from_afar(ctx, decision, ntri):
    """From afar a node's quantized bounds round together, so its unused slots
    are entered and pushed too; a ray without numbers enters every box.  The
    rows that only the used slots would need are not enough then.  The trees
    have at most six levels, whose 18 entries the default 19 rows hold."""
    sd = ra.generate_scene(ra.scene_params(api.RCH_SCENE_SOUP, seed=3, tri_count=ntri))
    r = np.random.default_rng(ntri)
    v = np.array([3.0, 2.0, 1.0]) + 1e-3 * (r.random((ntri, 1, 3)) + r.uniform(-0.2, 0.2, (ntri, 3, 3)))
    sd.vertices = np.ascontiguousarray(v.reshape(ntri, 9), np.float32)
    nodes, ordered, _, _ = ra.build_bvh(sd.vertices)
    s = ctx.upload(sd, nodes, ordered)
    n = 4096
    target = v.reshape(-1, 3)[r.integers(0, 3 * ntri, n)]
    d = r.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    rays = api.make_rays((target - d * r.uniform(1e2, 2e4, (n, 1))).astype(np.float32), d.astype(np.float32))
    f = rays.view(np.float32).reshape(n, 8)
    f[5::64, 0:3] = np.nan
    f[6::64, 4:7] = np.nan
    f[7::64, 0] = np.inf
    try:
        results = {}
        for rows in (0, *range(1, 19), 1):
            ctx.set_tuning(stack_limit=rows)
            hits = ctx.trace_closest(s, rays)
            outgrown = ctx.stats().overflow_rays
            results[rows] = hits.tobytes(), np.asarray(ctx.trace_any(s, rays)).tobytes(), outgrown
    finally:
        ctx.set_tuning()
        s.close()
    assert results[0][2] == 0
    for rows, got in results.items():
        assert got[:2] == results[0][:2], rows
    if ntri <= 10:  # one node with an unused slot: two entries if only the used ones counted
        assert results[2][2] > 0
