"""Host arrays to the device and back, and queries of host arrays, at the
edges of what goes through the context's page-locked chunks (2 MiB down, up to
512 KiB up, up to 65,536 rays of a query)."""
import ctypes as C

import numpy as np
import pytest

import raycer_amd as ra
from raycer_amd import api
from tests.helpers import random_rays

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.mark.parametrize("offset", [0, 3])
@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("n", [1, 63, MB // 2, MB // 2 + 1, 2 * MB - 1, 2 * MB, 2 * MB + 1, 4 * MB, 4 * MB + 129, 9 * MB + 5])
def test_round_trip(ctx, n, pinned, offset):
    data = np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8)
    blocks = [ctx.pinned(n + offset + 64, np.uint8) for _ in range(2)] if pinned else []
    src, dst = [b.array for b in blocks] if pinned else [np.zeros(n + offset + 64, np.uint8) for _ in range(2)]
    src[offset:offset + n] = data
    p = C.c_void_p()
    api.check(api.lib().rc_device_alloc(ctx.h, n, C.byref(p)))
    try:
        for _ in range(2):  # the chunks are used again
            dst[:] = 0
            api.check(api.lib().rc_memcpy_h2d(ctx.h, p, src.ctypes.data + offset, n))
            api.check(api.lib().rc_memcpy_d2h(ctx.h, dst.ctypes.data + offset, p, n))
            assert np.array_equal(dst[offset:offset + n], data)
            assert not dst[:offset].any() and not dst[offset + n:].any()
    finally:
        api.check(api.lib().rc_device_free(ctx.h, p))
        del src, dst
        for b in blocks:
            b.close()


@pytest.mark.parametrize("n", [1, 65535, 65536, 65537])
def test_host_queries_equal_device_queries(ctx, n):
    sd = ra.generate_scene(ra.scene_params(api.RCH_SCENE_SOUP, seed=5, tri_count=2000))
    nodes, ordered, _, _ = ra.build_bvh(sd.vertices)
    s = ctx.upload(sd, nodes, ordered)
    v = sd.vertices.reshape(-1, 3)
    rays = random_rays(n, 9, v.min(0), v.max(0))
    hits, occ = np.empty((n, 4), np.float32), np.empty(n, np.uint8)
    lib, bufs = api.lib(), []
    for nbytes in (rays.nbytes, hits.nbytes, occ.nbytes):
        p = C.c_void_p()
        api.check(lib.rc_device_alloc(ctx.h, nbytes, C.byref(p)))
        bufs.append(p)
    try:
        api.check(lib.rc_memcpy_h2d(ctx.h, bufs[0], rays.ctypes.data, rays.nbytes))
        api.check(lib.rc_trace_closest_device(ctx.h, s.h, bufs[0], n, bufs[1]))
        api.check(lib.rc_trace_any_device(ctx.h, s.h, bufs[0], n, bufs[2]))
        api.check(lib.rc_memcpy_d2h(ctx.h, hits.ctypes.data, bufs[1], hits.nbytes))
        api.check(lib.rc_memcpy_d2h(ctx.h, occ.ctypes.data, bufs[2], occ.nbytes))
        assert ctx.trace_closest(s, rays).tobytes() == hits.tobytes()
        assert np.asarray(ctx.trace_any(s, rays)).tobytes() == occ.tobytes()
    finally:
        for p in bufs:
            api.check(lib.rc_device_free(ctx.h, p))
        s.close()
