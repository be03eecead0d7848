"""The Phong raycast at the edges of its 32x8 blocks, with stacks that spill or
are walked again, into pageable, page-locked and unaligned arrays: always the
same bits, and the hits those of the ray queries for the same rays."""
import numpy as np
import pytest

import raycer_amd as ra
from raycer_amd import api

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
