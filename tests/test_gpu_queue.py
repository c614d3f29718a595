"""Render queues in segments: path counts around the steps of a block and of a round of
blocks over the segments, where a segment is empty, partial or full."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# paths: 1 short block; 1 full; 1 and 2 over; 4 full; 1 past; 8 and a bit; many, ragged
SIZES = [(5, 4, 1), (16, 16, 1), (43, 6, 1), (32, 32, 1), (25, 41, 1), (47, 15, 3), (61, 37, 8)]


@pytest.mark.parametrize("w,h,spp", SIZES)
def test_reference_render_matches_oracle(tt, oracle, ctx, w, h, spp):
    from trenchanttracer_amd import workloads
    print(f"queue segments, reference mode: {w}x{h}x{spp}", file=sys.stderr, flush=True)
    mesh, mats, cam = workloads.cornell(subdiv=2, width=w, height=h)
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh, mats)
    img, _ = scene.render(cam, tt.render_params(spp=spp, max_depth=6, seed=3, mode=tt.RENDER_REFERENCE))
    want = oracle.render_ref(oracle.CompactBVH(bvh.export_compact()), mesh.arrays(), mats, cam, spp=spp, max_depth=6,
                             seed=3, env=None)
    assert np.array_equal(img.view(np.int32), want.view(np.int32))
    scene.close()


@pytest.mark.parametrize("w,h,spp", SIZES)
def test_path_render_does_not_depend_on_the_passes(tt, ctx, w, h, spp):
    """All samples in one pass, one sample per pass, and a graph of one: the same image and
    ray counts."""
    from trenchanttracer_amd import workloads
    print(f"queue segments, path mode: {w}x{h}x{spp}", file=sys.stderr, flush=True)
    mesh, mats, cam = workloads.cornell(subdiv=2, width=w, height=h)
    scene = tt.DeviceScene(ctx, mesh, tt.BVH.build(mesh), mats)
    out = []
    for kw in (dict(), dict(paths_in_flight=w * h), dict(paths_in_flight=w * h, use_graph=True),
               dict(refill=8, refill_camera=16, block=256)):
        img, st = scene.render(cam, tt.render_params(spp=spp, max_depth=7, rr_depth=2, seed=4, mode=tt.RENDER_PATH, **kw))
        out.append((img.view(np.int32), st["rays_extension"], st["rays_shadow"]))
        assert np.isfinite(img).all() and img.max() > 0
    for got in out[1:]:
        assert np.array_equal(got[0], out[0][0]) and got[1:] == out[0][1:]
    scene.close()


@pytest.mark.parametrize("spp", [1, 8, 9, 16, 17, 32, 33, 70])
def test_sample_sums_match_oracle_and_passes(tt, oracle, ctx, spp):
    """Samples per pass around the chunks a block of pixels is summed in, on pixel counts
    that leave a partial block."""
    from trenchanttracer_amd import workloads
    print(f"sample sums: {spp} samples", file=sys.stderr, flush=True)
    for w, h in ((9, 8), (29, 9)):
        mesh, mats, cam = workloads.cornell(subdiv=1, width=w, height=h)
        bvh = tt.BVH.build(mesh)
        scene = tt.DeviceScene(ctx, mesh, bvh, mats)
        img, _ = scene.render(cam, tt.render_params(spp=spp, max_depth=4, seed=6, mode=tt.RENDER_REFERENCE))
        want = oracle.render_ref(oracle.CompactBVH(bvh.export_compact()), mesh.arrays(), mats, cam, spp=spp,
                                 max_depth=4, seed=6, env=None)
        assert np.array_equal(img.view(np.int32), want.view(np.int32))
        prm = dict(spp=spp, max_depth=4, rr_depth=2, seed=7, mode=tt.RENDER_PATH)
        for fp64 in (False, True):
            a = scene.render(cam, tt.render_params(fp64=fp64, **prm))[0]
            b = scene.render(cam, tt.render_params(fp64=fp64, paths_in_flight=w * h, **prm))[0]
            assert np.array_equal(a.view(np.int32), b.view(np.int32)) and a.max() > 0
        scene.close()
