"""Trace calls of more than 2^30 rays: in the caller's order (several launches) and in
Morton order (one), against the records of their repeated pattern."""
import ctypes as C
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_more_than_2_to_the_30_rays(tt):
    from trenchanttracer_amd import _native as N
    ctx = tt.Context(0)   # its own, which gives the sort's workspace back
    n, m = (1 << 30) + 70_001, 1 << 18
    mesh = tt.Mesh.soup(3000, seed=6, mu=float(np.log(0.05)))
    scene = tt.DeviceScene(ctx, mesh, tt.BVH.build(mesh))
    base = tt.rays_incoherent(mesh, m, seed=8)
    want = np.stack([x.view(np.int32) for x in scene.intersect(base)], 1)
    hit = scene.occluded(base)
    rays = tt.DeviceBuffer(ctx, n * 32)   # 34 GB, and the workspace of the sort 18 GB
    rays.upload(base)
    have = m
    while have < n:   # the pattern again and again
        more = min(have, n - have)
        tt.check(N.lib.tt_dev_copy(ctx._h, C.c_void_p(rays.ptr + have * 32), C.c_void_p(rays.ptr), more * 32))
        have += more
    for any_hit, ref in ((False, want), (True, hit)):
        out = tt.DeviceBuffer(ctx, (n + 64) * ref.itemsize * (ref.size // m))
        for reorder in (0, 1):
            print(f"{n} rays, any hit {any_hit}, reorder {reorder}", file=sys.stderr, flush=True)
            out.zero()
            trace = scene.trace_any if any_hit else scene.trace_closest
            trace(rays, n, out, tt.trace_cfg(0, 16, 128, reorder=reorder))
            ctx.sync()
            # the ends, both sides of 2^30, and between (the pattern's length divides 2^30)
            for at in [0, (1 << 30) - m, 1 << 30] + [m * k for k in range(100, 4096, 371)]:
                k = min(m, n - at)
                got = np.empty((k,) + ref.shape[1:], np.int32)
                tt.check(N.lib.tt_memcpy_d2h(ctx._h, C.c_void_p(got.ctypes.data),
                                             C.c_void_p(out.ptr + at * got[0].nbytes), got.nbytes))
                assert np.array_equal(got, ref[:k]), at
            end = np.empty((64,) + ref.shape[1:], np.int32)
            tt.check(N.lib.tt_memcpy_d2h(ctx._h, C.c_void_p(end.ctypes.data),
                                         C.c_void_p(out.ptr + n * end[0].nbytes), end.nbytes))
            assert not end.any()
        out.free()
    rays.free()
    scene.close()
    ctx.close()
