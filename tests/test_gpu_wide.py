"""The four-child walk against the oracle's two-child one where its rounding, ties and
limits can show: rays along axes and box faces, through shared edges and vertices, exact
ties between coincident triangles, leaves too large for a node's offsets, origins far
away, non-finite and degenerate rays, and short and deep stacks."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grid(n, z, rng=None):
    """n x n unit quads in the plane z as two triangles each (shared edges and corners)."""
    v, t = [], []
    for y in range(n + 1):
        for x in range(n + 1):
            v.append([x, y, z if rng is None else z + float(rng.normal(0.0, 0.3))])
    for y in range(n):
        for x in range(n):
            a = y * (n + 1) + x
            t += [[a, a + 1, a + n + 2], [a, a + n + 2, a + n + 1]]
    return np.array(v, np.float32), np.array(t, np.int32)


def _join(parts):
    v, t, at = [], [], 0
    for pv, pt in parts:
        v.append(pv)
        t.append(pt + at)
        at += len(pv)
    return np.concatenate(v), np.concatenate(t)


def _mesh(tt, kind):
    rng = np.random.default_rng(3)
    if kind == "layers":         # flat boxes, shared edges, rays along the planes' axes
        return tt.Mesh.from_arrays(*_join([_grid(16, float(z)) for z in range(12)]))
    if kind == "hills":
        return tt.Mesh.from_arrays(*_join([_grid(24, 3.0 * z, rng) for z in range(6)]))
    if kind == "coincident":     # every triangle four times: exact ties throughout
        v, t = _grid(20, 1.0, rng)
        v2, t2 = _grid(20, 4.0, rng)
        return tt.Mesh.from_arrays(*_join([(v, np.concatenate([t] * 4)), (v2, t2)]))
    if kind in ("piles", "spread"):   # 60 coincident triangles at each place: large leaves
        n = 200 if kind == "piles" else 12000   # (a tree past the packed records' size)
        v = rng.normal(0, 4, (n, 1, 3)) + rng.normal(0, 2 if n == 200 else 0.2, (n, 3, 3))
        v = np.repeat(v, 60, axis=0).reshape(-1, 3)
        return tt.Mesh.from_arrays(v.astype(np.float32), np.arange(len(v), dtype=np.int32).reshape(-1, 3))
    if kind == "line":           # triangles along a line: a deep tree, many pending children
        c = np.geomspace(1.0, 4096.0, 3000)[:, None, None] * np.array([1.0, 1e-3, 1e-3])
        v = c + rng.normal(0, 1, (3000, 3, 3)) * (0.05 * c[:, :, :1])
        return tt.Mesh.from_arrays(v.reshape(-1, 3).astype(np.float32), np.arange(9000, dtype=np.int32).reshape(-1, 3))
    raise ValueError(kind)


def _rays(mesh, seed):
    rng = np.random.default_rng(seed)
    a = mesh.arrays()
    v = a["verts"].astype(np.float64)
    lo, hi = v.min(0), v.max(0)
    ext = np.maximum(hi - lo, 1e-3)
    out = []

    def add(o, d, tmin=0.0, tmax=1e20):
        r = np.zeros((len(o), 8), np.float32)
        r[:, :3], r[:, 3], r[:, 4:7], r[:, 7] = o, tmin, d, tmax
        out.append(r)
    n = 3000
    inside = lo + rng.random((n, 3)) * ext
    d = rng.normal(size=(n, 3))
    add(inside, d / np.linalg.norm(d, axis=1, keepdims=True))
    add(inside, d * 1e-6, 1e-4, 1e30)
    # aimed exactly at vertices and edge midpoints
    tri = a["tris"][rng.integers(len(a["tris"]), size=n)]
    eye = lo - 2.0 * ext + rng.random((n, 3)) * 5.0 * ext
    add(eye, v[tri[:, 0]] - eye)
    add(eye, 0.5 * (v[tri[:, 0]] + v[tri[:, 1]]) - eye)
    # along the axes (both signs, zero and negative-zero components), through vertices
    for k in range(3):
        for s in (1.0, -1.0):
            ax = np.zeros((n // 2, 3), np.float32)
            ax[:, k] = s
            ax[::3, (k + 1) % 3] = -0.0
            o = v[tri[:n // 2, 1]].copy()
            o[:, k] = lo[k] - 1.0 if s > 0 else hi[k] + 1.0
            add(o, ax)
    # starting on a vertex, in a plane of the geometry
    flat = d.copy()
    flat[:, 2] = 0.0
    add(v[tri[:, 2]], flat, 1e-4)
    # far origins, infinite reach, nothing to reach, negative starts
    add(eye * 1e4, v[tri[:, 0]] - eye * 1e4, 0.0, np.inf)
    add(inside, d, 0.5, 0.25)
    add(inside[:500], d[:500], -1.0)
    add(inside[:500], d[:500], -0.0)
    add(inside[:500], d[:500], 0.0, 0.0)
    # degenerate and non-finite rays
    odd = np.array([np.nan, np.inf, -np.inf, 0.0, 1e38, 1e-40])
    o, e = inside[:600].copy(), d[:600].copy()
    o[np.arange(300), rng.integers(3, size=300)] = rng.choice(odd, 300)
    e[np.arange(300, 600), rng.integers(3, size=300)] = rng.choice(odd, 300)
    e[590:] = 0.0
    add(o, e)
    add(inside[:6], d[:6], odd, 1e20)
    add(inside[:6], d[:6], 0.0, odd)
    return np.concatenate(out)


@pytest.mark.parametrize("kind", ["layers", "hills", "coincident", "piles", "line", "spread"])
def test_four_child_walk_matches_oracle(tt, oracle, ctx, kind):
    print(f"four-child walk: {kind}", file=sys.stderr, flush=True)
    mesh = _mesh(tt, kind)
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh)
    rays = _rays(mesh, 5)
    cb = oracle.CompactBVH(bvh.export_compact())
    want, _ = cb.trace(rays)
    any_want, _ = cb.trace(rays, any_hit=True)
    hit = (oracle.hit_ids(any_want) >= 0).astype(np.int32)
    for cfg in (None, tt.trace_cfg(0, 8, 64, refill=16), tt.trace_cfg(1, 32, 256, refill=1, reorder=1),
                tt.trace_cfg(1, 16, 128), tt.trace_cfg(1, 8, 64, refill=16)):
        got = scene.intersect(rays, cfg)
        for k, (x, name) in enumerate(zip(got, ("id", "t", "u", "v"))):
            bad = np.flatnonzero(x.view(np.int32) != want[:, k].view(np.int32))
            assert len(bad) == 0, f"{kind}: {len(bad)} {name}, first ray {bad[0]}: {rays[bad[0]]}"
        flags = scene.occluded(rays, cfg)
        bad = np.flatnonzero(flags != hit)
        assert len(bad) == 0, f"{kind}: {len(bad)} flags, first ray {bad[0]}: {rays[bad[0]]}"
    scene.close()


@pytest.mark.parametrize("seed,tris,size", [(2, 400, 5.0), (13, 400, 20.0), (14, 100, 10.0), (15, 2000, 5.0)])
def test_variant_0_is_exact_for_hits_of_rounding_noise(tt, oracle, ctx, seed, tris, size):
    """Rays almost in the planes of large triangles, whose computed distances can lie far
    from them: the records of the single-lane order."""
    print(f"grazing rays: {tris} triangles of size {size}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(seed)
    v = (rng.uniform(-10, 10, (tris, 1, 3)) + rng.normal(0, size, (tris, 3, 3))).astype(np.float32)
    mesh = tt.Mesh.from_arrays(v.reshape(-1, 3), np.arange(3 * tris, dtype=np.int32).reshape(-1, 3))
    bvh = tt.BVH.build(mesh)
    scene = tt.DeviceScene(ctx, mesh, bvh)
    n = 1_000_000
    k = rng.integers(tris, size=n)
    w = rng.dirichlet((1, 1, 1), n)
    t = v[k].astype(np.float64)
    p = (t * w[:, :, None]).sum(1)
    e1, e2 = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    nn = np.cross(e1, e2)
    nn /= np.linalg.norm(nn, axis=1, keepdims=True)
    a = rng.uniform(0, 2 * np.pi, n)
    u = e1 / np.linalg.norm(e1, axis=1, keepdims=True)
    off = 10 ** rng.uniform(-8, -2, n) * rng.choice([-1, 1], n)
    d = u * np.cos(a)[:, None] + np.cross(nn, u) * np.sin(a)[:, None] + nn * off[:, None]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3] = p - d * (10 ** rng.uniform(-2, 1.5, n))[:, None]
    rays[:, 4:7], rays[:, 7] = d, 1e20
    want, _ = oracle.CompactBVH(bvh.export_compact()).trace(rays, nthreads=8)
    for cfg in (None, tt.trace_cfg(0, 16, 256, refill=16)):
        for j, x in enumerate(scene.intersect(rays, cfg)):
            assert np.array_equal(x.view(np.int32), want[:, j].view(np.int32))
    scene.close()


def test_four_child_walk_of_several_trees(tt, ctx):
    """Scenes of a batch (one node array, per-scene roots), one of them below the cost at
    which a scene of its own gets a four-child tree: each image equals its own render's."""
    from trenchanttracer_amd import workloads
    meshes, mats, cams, env, _ = workloads.batched(n=3, seed=5, tri_lo=300, tri_hi=4000, resolutions=(48,))
    # no emitters: a batch's next-event estimation samples all its scenes' lights
    meshes.append(tt.Mesh.soup(30, seed=4, mu=float(np.log(0.3))))
    mats.append([tt.material(tt.MAT_DIFFUSE, (0.6, 0.7, 0.8))])
    cams.append(tt.camera((0.5, 0.5, -1.2), (0.0, 0.0, 1.0), fov=(50.0, 50.0), width=48, height=40))
    bvhs = [tt.BVH.build(m) for m in meshes]
    prm = tt.render_params(spp=4, max_depth=6, rr_depth=3, seed=2, mode=tt.RENDER_PATH)
    batch = tt.Batch(ctx, meshes, bvhs, mats, env=env)
    imgs, _ = batch.render(cams, prm)
    for m, b, mm, c, im in zip(meshes, bvhs, mats, cams, imgs):
        s = tt.DeviceScene(ctx, m, b, mm, env=env)
        one, _ = s.render(c, prm)
        assert np.array_equal(one.view(np.int32), im.view(np.int32))
        s.close()
    batch.close()


@pytest.mark.parametrize("tris", [30, 20000])   # two-child loop, four-child walk
def test_few_rays_in_small_groups(tt, ctx, tris):
    """Counts around the steps of the group size (1 to 64 rays): the records of a launch of
    full groups, and nothing written past the end."""
    mesh = tt.Mesh.soup(tris, seed=4, mu=float(np.log(0.3))) if tris == 30 else tt.Mesh.soup(tris, seed=6)
    scene = tt.DeviceScene(ctx, mesh, tt.BVH.build(mesh))
    total = 200_003
    d = tt.DeviceBuffer.from_array(ctx, tt.rays_incoherent(mesh, total, seed=8))
    h = tt.DeviceBuffer(ctx, (total + 64) * 16)
    f = tt.DeviceBuffer(ctx, (total + 64) * 4)

    def trace(n, cfg):
        h.upload(np.full((n + 64, 4), 7.0, np.float32))
        f.upload(np.full(n + 64, 7, np.int32))
        scene.trace_closest(d, n, h, cfg)
        scene.trace_any(d, n, f, cfg)
        ctx.sync()
        return h.download((n + 64, 4), np.int32), f.download(n + 64, np.int32)
    want, hit = trace(total, None)
    for n in (1, 2, 63, 64, 65, 2047, 2048, 2049, 4096, 4097, 65_535, 65_537, 131_072, 131_073):
        print(f"small groups: {n} rays", file=sys.stderr, flush=True)
        for cfg in (None, tt.trace_cfg(1, 8, 256), tt.trace_cfg(0, 16, 64, refill=24), tt.trace_cfg(1, 16, 64, reorder=1)):
            got, flags = trace(n, cfg)
            assert np.array_equal(got[:n], want[:n]) and np.array_equal(flags[:n], hit[:n])
            assert (got[n:].view(np.float32) == 7.0).all() and (flags[n:] == 7).all()
    for b in (d, h, f):
        b.free()
    scene.close()


def test_sweeps_trace_every_ray_once(tt, ctx):
    """refill 0 traces the range in parts; ray counts below, at and past one group per
    resident wave and one part, ragged: the records of the persistent launch, and nothing
    written past the end."""
    mesh = tt.Mesh.soup(20000, seed=6)
    scene = tt.DeviceScene(ctx, mesh, tt.BVH.build(mesh))
    rays = tt.rays_incoherent(mesh, 3_000_017, seed=7)
    d = tt.DeviceBuffer.from_array(ctx, rays)
    h = tt.DeviceBuffer(ctx, (len(rays) + 64) * 16)

    def trace(n, cfg):
        h.upload(np.full((n + 64, 4), 7.0, np.float32))
        scene.trace_closest(d, n, h, cfg)
        ctx.sync()
        return h.download((n + 64, 4), np.int32)
    for n in (65_537, 327_681, 393_217, 700_001, 1_572_863, 1_572_865, 3_000_017):
        print(f"sweeps: {n} rays", file=sys.stderr, flush=True)
        for block in (64, 256):
            got = trace(n, tt.trace_cfg(0, 16, block))
            assert np.array_equal(got, trace(n, tt.trace_cfg(0, 16, block, refill=8)))
            assert (got[n:].view(np.float32) == 7.0).all()
    d.free()
    h.free()
    scene.close()
