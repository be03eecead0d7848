"""The Phong raycast at the edges of its 32x8 blocks, with stacks that spill or
are walked again, into pageable, page-locked and unaligned arrays: always the
same bits, and the hits those of the ray queries for the same rays."""
import numpy as np
import pytest

import raycer_amd as ra
from raycer_amd import api
from tests.helpers import overlapping_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(2, 2), (31, 9), (32, 8), (33, 7), (161, 95)])
def test_phong_variants_agree(ctx, decision, width, height):
    sd = ra.generate_scene(ra.scene_params(api.RCH_SCENE_SPHERE_GROUND, seed=1, level=4, grid=64))
    nodes, ordered, _, _ = ra.build_bvh(sd.vertices)
    s = ctx.upload(sd, nodes, ordered)
    n = width * height
    args = (s, sd.desc.camera, width, height, 7, sd.desc.cfg.ray_start_offset, sd.desc.light)
    blocks = [ctx.pinned(n * size + 64, np.uint8) for size in (4, 4, 16)]

    def views(offset):
        a = [b.array[offset:] for b in blocks]
        return [a[0][:4 * n].view(np.int32), a[1][:4 * n].view(np.float32), a[2][:16 * n].view(np.float32).reshape(n, 4)]

    try:
        ref = [x.tobytes() for x in ctx.raycast_phong(*args)]
        assert (np.frombuffer(ref[0], np.int32) >= 0).any()
        for offset in (0, 4):  # 16-byte aligned colours, and not
            for b in blocks:
                b.array[:] = 0xA5
            out = ctx.raycast_phong(*args, out=views(offset))
            assert [x.tobytes() for x in out] == ref
            for b, x in zip(blocks, out):
                assert (b.array[:offset] == 0xA5).all() and (b.array[offset + x.nbytes:] == 0xA5).all()
        for limit in (1, 4, 6):
            ctx.set_tuning(stack_limit=limit)
            assert [x.tobytes() for x in ctx.raycast_phong(*args)] == ref
    finally:
        ctx.set_tuning()
        out = None
        for b in blocks:
            b.close()
        s.close()


# At most as many pixels as there are spill slots (2,048), but more traversals
# than that outgrow their rows: a pixel's primary and shadow ray each claim a
# slot, so pixels are listed and walked again.  The light is at the camera:
# most shadow rays reach it, and a pixel left out would lack its light.
@pytest.mark.parametrize("width,height", [(45, 45), (32, 64)])
@pytest.mark.parametrize("limit", [4, 5])
def test_phong_loses_no_listed_pixel(ctx, decision, width, height, limit):
    sd = overlapping_scene()
    nodes, ordered, _, _ = ra.build_bvh(sd.vertices)
    s = ctx.upload(sd, nodes, ordered)
    light = api.PointLight((0.5, 0.5, 0.5), (1.0, 1.0, 1.0), 1.0, 1000.0, 1.0, (1.0, 1.0, 1.0), 0.1)
    args = (s, sd.desc.camera, width, height, 7, sd.desc.cfg.ray_start_offset, light)
    try:
        ctx.set_tuning(stack_limit=1)
        ref = [x.tobytes() for x in ctx.raycast_phong(*args)]
        ctx.set_tuning(stack_limit=limit)
        assert [x.tobytes() for x in ctx.raycast_phong(*args)] == ref
    finally:
        ctx.set_tuning()
        s.close()
    assert (np.frombuffer(ref[2], np.float32)[::4] > 0.1).mean() > 0.5  # ambient alone gives less
