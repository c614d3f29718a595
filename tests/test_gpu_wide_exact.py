"""The four-child closest-hit walk where a record depends on one comparison: segments that
end exactly on a surface, against the oracle's single-lane walk."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CFGS = ((0, 16, 128, 0, 0), (0, 8, 64, 16, 0), (1, 16, 256, 32, 1), (1, 16, 64, 0, 0))


def _say(msg):
    print(msg, file=sys.stderr, flush=True)


def _check(tt, oracle, scene, bvh, rays, what, cfgs=CFGS):
    cb = oracle.CompactBVH(bvh.export_compact())
    want, _ = cb.trace(rays, nthreads=8)
    for c in cfgs:
        cfg = tt.trace_cfg(*c[:3], refill=c[3], reorder=c[4])
        for k, (x, name) in enumerate(zip(scene.intersect(rays, cfg), ("id", "t", "u", "v"))):
            bad = np.flatnonzero(x.view(np.int32) != want[:, k].view(np.int32))
            assert len(bad) == 0, f"{what}, {c}: {len(bad)} {name}, first ray {bad[0]}: {rays[bad[0]]}"
    return want


def _soup_over_plane(tt):
    """20000 triangles in the unit cube (enough for the four-child tree) over the plane z = 0
    from -0.5 to 1.5, tessellated in right triangles with legs of 0.25 (front faces up)."""
    soup = tt.Mesh.soup(20000, seed=6, mu=float(np.log(0.03))).arrays()
    x, y = np.meshgrid(np.arange(-2, 7) * 0.25, np.arange(-2, 7) * 0.25)
    v = np.stack([x.ravel(), y.ravel(), np.zeros(x.size)], 1)
    a = (np.arange(8)[:, None] * 9 + np.arange(8)).ravel()
    t = np.concatenate([np.stack([a, a + 1, a + 9], 1), np.stack([a + 10, a + 9, a + 1], 1)])
    return tt.Mesh.from_arrays(np.concatenate([soup["verts"], v]).astype(np.float32),
                               np.concatenate([soup["tris"], t + len(soup["verts"])]).astype(np.int32))


def test_segments_ending_on_a_surface(tt, oracle, ctx):
    """A triangle exactly at tmax is no hit, one unit in the last place before it is: rays
    down to the plane, and rays retraced to the distance of their own hit."""
    mesh = _soup_over_plane(tt)
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh)
    rng = np.random.default_rng(1)
    n = 4000
    down = np.zeros((n, 8), np.float32)
    # beside the cube nothing lies before the plane; over it, mostly
    down[:, :2] = rng.integers(-4, 12, (n, 2)) / 8.0 + 0.03125
    down[:3 * n // 4, 0] = -np.abs(down[:3 * n // 4, 0] % 0.375) - 0.0625
    down[:, 2] = down[:, 7] = rng.choice([0.25, 0.5, 1.0, 2.0, 5.0], n)
    down[:, 6] = -1.0
    free = np.concatenate([tt.rays_incoherent(mesh, 20000, seed=3),
                           tt.rays_primary(160, 120, 1, (0.5, 0.5, 3.0), (0.5, 0.5, 0.0), seed=3), down])
    free[-n:, 7] = 1e20
    _say("segments ending on a surface: reaching further")
    t = _check(tt, oracle, scene, bvh, free, "reaching further")[:, 1].copy()
    assert (t[-n:] == free[-n:, 2]).sum() > n // 2   # the plane is hit at the origin's height
    for name, end in (("on it", t), ("before it", np.nextafter(t, np.float32(0))),
                      ("past it", np.nextafter(t, np.float32(np.inf)))):
        _say(f"segments ending on a surface: {name}")
        rays = free.copy()
        rays[:, 7] = end
        _check(tt, oracle, scene, bvh, rays, name)
    scene.close()
