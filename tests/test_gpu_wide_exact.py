"""The four-child closest-hit walk where a record depends on one comparison or on rounding:
segments that end exactly on a surface, rays nearly in their triangles' planes, and the
scenes of test_gpu_wide.py at scales at which exact rays take that walk; against the
oracle's single-lane walk."""
import sys

import numpy as np
import pytest
import test_gpu_wide

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
    assert scene.walk()[0] and scene.walk()[1] > 0.0
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


EXACT = tuple(c for c in CFGS if c[0] == 0)


def _triangles(seed, tris, size, extent):
    """Random triangles in a cube, |e1| |e2| up to size^2."""
    rng = np.random.default_rng(seed)
    v = rng.uniform(-extent, extent, (tris, 1, 3)) + rng.normal(0, 1, (tris, 3, 3)) * size
    p = np.linalg.norm(v[:, 1] - v[:, 0], axis=1) * np.linalg.norm(v[:, 2] - v[:, 0], axis=1)
    c = v.mean(1, keepdims=True)
    return rng, (c + (v - c) * np.sqrt(np.minimum(1, 0.99 * size * size / p))[:, None, None]).astype(np.float32)


def _grazing(rng, v, n, near, far):
    """Rays at random points of the triangles v from near to far away, nearly in their
    planes: det from the 1e-5 it is accepted from to ten times that."""
    t = v[rng.integers(len(v), size=n)].astype(np.float64)
    p = (t * rng.dirichlet((1, 1, 1), n)[:, :, None]).sum(1)
    e1, e2 = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    nn = np.cross(e1, e2)
    nn /= np.linalg.norm(nn, axis=1, keepdims=True)
    a = rng.uniform(0, 2 * np.pi, n)
    u = e1 / np.linalg.norm(e1, axis=1, keepdims=True)
    pr = np.linalg.norm(e1, axis=1) * np.linalg.norm(e2, axis=1)
    off = 1e-5 / pr * 10 ** rng.uniform(0, 1.0, n)
    d = u * np.cos(a)[:, None] + np.cross(nn, u) * np.sin(a)[:, None] - nn * off[:, None]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3] = p - d * (10 ** rng.uniform(np.log10(near), np.log10(far), n))[:, None]
    rays[:, 4:7], rays[:, 7] = d, 1e20
    return rays


# the last column: whether exact rays from within the scene take the four-child walk there
@pytest.mark.parametrize("seed,tris,size,extent,near,far,wide", [
    (2, 2000, 1.0, 4, 30, 1000, False), (3, 20000, 1.0, 10, 10, 1000, False),
    (4, 2000, 0.4, 0.5, 0.1, 10, False), (7, 20000, 0.1, 1, 0.1, 10, True), (8, 20000, 0.1, 1, 10, 1000, True),
    (9, 200000, 0.05, 1, 0.1, 10, True), (10, 20000, 0.05, 0.3, 0.01, 3, True), (11, 3000, 0.2, 0.5, 0.03, 3, True)])
def test_variant_0_is_exact_for_grazing_rays(tt, oracle, ctx, seed, tris, size, extent, near, far, wide):
    _say(f"grazing rays: {tris} triangles of size {size} in {extent}, {near} to {far} away")
    rng, v = _triangles(seed, tris, size, extent)
    mesh = tt.Mesh.from_arrays(v.reshape(-1, 3), np.arange(3 * tris, dtype=np.int32).reshape(-1, 3))
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh)
    assert scene.walk()[0] and (scene.walk()[1] > 0.0) == wide
    rays = _grazing(rng, v, 1_000_000, near, far)
    rays[::7, 4:7] *= 0.25   # lengths other than 1
    rays[1::7, 4:7] *= 3.0
    _check(tt, oracle, scene, bvh, rays, "grazing", EXACT)
    scene.close()


@pytest.mark.parametrize("kind,scale", [("layers", 2.0 ** -3), ("layers", 2.0 ** -5), ("hills", 2.0 ** -3),
                                        ("hills", 2.0 ** -5), ("coincident", 2.0 ** -4), ("piles", 2.0 ** -5),
                                        ("spread", 2.0 ** -4)])
def test_exact_four_child_walk_matches_oracle(tt, oracle, ctx, kind, scale):
    """test_gpu_wide.py's scenes and rays, small enough for exact rays to take the
    four-child walk."""
    _say(f"exact four-child walk: {kind} at {scale}")
    a = test_gpu_wide._mesh(tt, kind).arrays()
    mesh = tt.Mesh.from_arrays(a["verts"] * np.float32(scale), a["tris"])
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh)
    assert scene.walk()[1] > 0.0
    _check(tt, oracle, scene, bvh, test_gpu_wide._rays(mesh, 5), kind)
    scene.close()


@pytest.mark.parametrize("seed,tris,size,spread,fov", [(4, 30, 2.0, 0.0, 1e-5), (6, 100, 1.0, 0.0, 1e-6),
                                                       (8, 400, 0.6, 3e-6, 1e-5)])
def test_path_mode_variant_0_is_exact_for_grazing_rays(tt, ctx, seed, tris, size, spread, fov):
    """A camera almost in the plane of large triangles, whose two-sided test accepts any
    determinant but 0: the image of the same scene with a triangle far away, which leaves
    the rest of the tree (without spatial splits) as it is and makes the scene one whose
    rays take the two-child loop."""
    _say(f"grazing camera rays: {tris} triangles of size {size}")
    rng = np.random.default_rng(seed)
    centre = np.stack([rng.uniform(0, 20, tris), rng.uniform(-10, 10, tris), rng.normal(0, spread, tris)], 1)
    flat = centre[:, None] + rng.normal(0, 1, (tris, 3, 3)) * np.array([size, size, 1e-6])
    centre = np.stack([rng.uniform(0, 20, 3000), rng.uniform(-10, 10, 3000), rng.uniform(-10, 10, 3000)], 1)
    v = np.concatenate([flat, centre[:, None] + rng.normal(0, 0.3, (3000, 3, 3))]).reshape(-1, 3)
    rot, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    v = v @ rot.T
    mats = [tt.material(tt.MAT_DIFFUSE, (0.5, 0.5, 0.5), emission=(k + 1.0, float(k * k), 1.0)) for k in range(61)]
    cam = tt.camera(tuple(rot @ [-3.0, 0.3, 0.0]), tuple(rot @ [1.0, 0.013, 0.0]), up=tuple(rot @ [0.0, 0.0, 1.0]),
                    fov=(60.0, fov), width=2048, height=1024)
    prm = tt.render_params(spp=2, max_depth=1, seed=seed, mode=tt.RENDER_PATH, variant=0)
    images = []
    for away in (False, True):
        w = np.concatenate([v, [[-5e3, -5e3, -5e3], [-5001, -5e3, -5e3], [-5e3, -5001, -5e3]]]) if away else v
        t = np.arange(len(w), dtype=np.int32).reshape(-1, 3)
        mesh = tt.Mesh.from_arrays(w.astype(np.float32), t, tri_mats=(np.arange(len(t)) % 61).astype(np.int32))
        scene = tt.DeviceScene(ctx, mesh, tt.BVH.build(mesh, split_alpha=1e30), mats)
        assert scene.walk()[0] != away
        images.append(scene.render(cam, prm)[0])
        scene.close()
    assert (images[0] > 0).any(2).mean() > 0.2
    bad = (images[0] != images[1]).any(2).sum()
    assert bad == 0, f"{bad} pixels differ"


@pytest.mark.parametrize("kind,scale", [("layers", 2.0 ** -5), ("hills", 1.0), ("coincident", 2.0 ** -5)])
def test_very_long_directions(tt, oracle, ctx, kind, scale):
    """Directions up to 2^127 long, whose slab terms are denormal."""
    a = test_gpu_wide._mesh(tt, kind).arrays()
    mesh = tt.Mesh.from_arrays(a["verts"] * np.float32(scale), a["tris"])
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh)
    base = test_gpu_wide._rays(mesh, 5)
    longest = np.abs(base[:, 4:7]).max(1)
    base = base[np.isfinite(base).all(1) & (longest > 0) & (base[:, 3] >= 0)]
    longest = np.abs(base[:, 4:7]).max(1)
    for k in (60, 79, 100, 118, 124, 127):
        _say(f"very long directions: {kind} at {scale}, 2^{k}")
        rays = base.copy()
        rays[:, 4:7] = rays[:, 4:7] / longest[:, None] * np.float32(2.0 ** k)
        rays[:, 3], rays[:, 7] = 0.0, 1e20
        _check(tt, oracle, scene, bvh, rays, f"2^{k}")
        want, _ = oracle.CompactBVH(bvh.export_compact()).trace(rays, any_hit=True, nthreads=8)
        assert np.array_equal(scene.occluded(rays), (oracle.hit_ids(want) >= 0).astype(np.int32))
    scene.close()


@pytest.mark.parametrize("offset,wide", [(100.0, True), (1000.0, True), (30000.0, False)])
def test_scenes_far_from_the_origin(tt, oracle, ctx, offset, wide):
    """Coordinates large against the scene, whose rounding widens the four-child walk's
    boxes: the records of the single-lane order, and no such walk where that costs more
    than it gives."""
    _say(f"scene at {offset}")
    a = tt.Mesh.soup(20000, seed=6, mu=float(np.log(0.03))).arrays()
    near = tt.Mesh.from_arrays(a["verts"], a["tris"])
    mesh = tt.Mesh.from_arrays(a["verts"] + np.float32(offset), a["tris"])
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh)
    assert scene.walk()[0] == wide
    rays = np.concatenate([tt.rays_incoherent(near, 40000, seed=3),
                           tt.rays_primary(200, 200, 1, (0.5, 0.5, -1.0), (0.5, 0.5, 0.0), seed=3)])
    rays[:, :3] += np.float32(offset)
    _check(tt, oracle, scene, bvh, rays, "far from the origin", EXACT)
    scene.close()


def test_rays_from_far_away(tt, oracle, ctx):
    """Origins 1 to 10^7 scene sizes away, around the distances at which the culling margin
    and the walk change: variant 0's records and any hit's flags; variant 1's distances to
    rounding."""
    mesh = tt.Mesh.soup(20000, seed=6, mu=float(np.log(0.03)))
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh)
    rng = np.random.default_rng(1)
    n = 20000
    at, d = rng.random((n, 3)), rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    cb = oracle.CompactBVH(bvh.export_compact())
    for away in (1.0, 3.9, 4.1, 300.0, 1e3, 5e4, 1e5, 1e7):
        _say(f"rays from far away: {away}")
        rays = np.zeros((n, 8), np.float32)
        rays[:, :3], rays[:, 4:7], rays[:, 7] = at - d * away, d, 1e20
        want = _check(tt, oracle, scene, bvh, rays, f"{away} away", EXACT)
        hit, _ = cb.trace(rays, any_hit=True, nthreads=8)
        assert np.array_equal(scene.occluded(rays), (oracle.hit_ids(hit) >= 0).astype(np.int32))
        ids, t, _, _ = scene.intersect(rays, tt.trace_cfg(1, 16, 128))
        assert ((ids >= 0) == (oracle.hit_ids(want) >= 0)).all()
        # noise of a computed distance off grazing rays: 1e-5 of the way
        assert (np.abs(t - want[:, 1]) <= 1e-5 * want[:, 1]).mean() > 0.999
    scene.close()


@pytest.mark.parametrize("tris,mu,copies,flip", [(3000, 0.1, 2, False), (3000, 0.1, 3, True), (20000, 0.03, 2, True),
                                                 (20000, 0.03, 5, False)])
def test_coincident_triangles(tt, oracle, ctx, tris, mu, copies, flip):
    """Every triangle several times, in shuffled order, with or without every other copy
    facing the other way; large ones are split over several leaves. Exact ties are won by
    the first triangle visited."""
    _say(f"coincident triangles: {copies} of {tris}")
    a = tt.Mesh.soup(tris, seed=6, mu=float(np.log(mu))).arrays()
    t = np.concatenate([a["tris"][:, ::-1] if flip and k % 2 else a["tris"] for k in range(copies)])
    t = t[np.random.default_rng(1).permutation(len(t))]
    mesh = tt.Mesh.from_arrays(a["verts"], np.ascontiguousarray(t))
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh)
    assert scene.walk()[0]
    rays = np.concatenate([tt.rays_incoherent(mesh, 60000, seed=3),
                           tt.rays_primary(200, 200, 1, (0.5, 0.5, -1.0), (0.5, 0.5, 0.0), seed=3)])
    want = _check(tt, oracle, scene, bvh, rays, "coincident")
    assert (oracle.hit_ids(want) >= 0).mean() > 0.3
    scene.close()
