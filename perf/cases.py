"""The work a user of this package has it do, as timed cases over its public entry points.

Each case is a dict of plain values; prepare() builds what a user's program holds before
the call (scene on the GPU, rays, network, cameras), run() is one call sequence of such a
program, work() the bytes and operations it cannot do without, exact() the result in
64 bits where plain torch can give it. Geometry and trees are built once per process (a
program keeps its tree, or loads it from its cache file); the device scene, the rays, the
random streams and the training rows come from the seed."""
import functools
import math

import numpy as np
import torch

import trenchanttracer_amd as tt
from trenchanttracer_amd import workloads

DEV = "cuda:0"
GEO_SEED = 1
EYE = (0.5, 0.5, -1.0)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # Picking under a cursor: a handful of rays in host memory through the host-buffer
        # call, where launches, copies and waits are everything.
        dict(name="pick_host_256", kind="intersect", tris=20_000, w=16, h=8, spp=1, scattered=128, variant=0),
        # Device buffers with the default configuration: one 720p frame of camera rays and
        # as many rays from surfaces.
        dict(name="closest_default_720p", kind="closest", tris=250_000, w=1280, h=720, spp=1, scattered=921_600,
             variant=0, block=128, refill=0, reorder=0),
        # The traversal benchmark: 1M triangles, 1080p x 2 camera rays and as many
        # incoherent ones, in the configuration the tuner picks.
        dict(name="closest_tuned_1m", kind="closest", tris=1_000_000, w=1920, h=1080, spp=2, scattered=4_147_200,
             variant=1, block=256, refill=32, reorder=1),
        # Shadow rays from surface points towards a light, default configuration.
        dict(name="occluded_default_1m", kind="any", tris=100_000, rays=1_000_003, variant=0, block=128, refill=0),
        # The reference-semantics image of the Cornell box with a mesh sphere.
        dict(name="reference_cornell_256", kind="reference", subdiv=4, w=256, h=256, spp=16, depth=8),
        # The interactive viewer: one sample per pixel and frame of the analytic Cornell
        # scene, accumulated and converted for display (four frames after a camera move).
        dict(name="viewer_640x360", kind="viewer", subdiv=3, w=640, h=360, frames=4, depth=10),
        # Path tracing a small closed room: short launches, many bounces.
        dict(name="path_room_256", kind="path", scene="room", subdiv=0, w=256, h=256, spp=64, depth=12),
        # Path tracing at full size: 1.31M triangles, mixed materials, sky with sun, 1080p,
        # 64 samples per pixel, 16 bounces.
        dict(name="path_1080p_64spp", kind="path", scene="sky", subdiv=8, w=1920, h=1080, spp=64, depth=16),
        # Several scenes of mixed size in one wavefront.
        dict(name="batch_8_scenes", kind="batch", scenes=8, tri_lo=1_000, tri_hi=150_000, res=512, spp=16, depth=8),
        # Learned path guiding: the network trains online between passes that grow 8x.
        dict(name="guided_online_540p", kind="guided", subdiv=6, w=960, h=540, spp=24, depth=12, paths=32_768,
             batch=65_536, bounces=1),
        # The guiding network: forward over an odd row count, and one Adam step.
        dict(name="guide_forward_70001", kind="guide_forward", rows=70_001),
        dict(name="guide_train_262144", kind="guide_train", rows=262_144),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["intersect", "closest", "closest", "any", "reference", "viewer", "path", "path", "batch",
                       "guided", "guide_forward", "guide_train"])
    if kind in ("intersect", "closest"):
        w = _log(rng, 8, 1920 if kind == "closest" else 640)
        h = max(2, int(w * rng.uniform(0.4, 1.0)))
        case = dict(kind=kind, tris=_log(rng, 1_000, 400_000), w=w, h=h, spp=1, scattered=_log(rng, 64, 2 * w * h + 64),
                    variant=rng.choice([0, 1]))
        if kind == "closest":
            case |= dict(block=rng.choice([64, 128, 256]), refill=rng.choice([0, 16, 32]), reorder=rng.choice([0, 1]))
        return case
    if kind == "any":
        return dict(kind=kind, tris=_log(rng, 1_000, 400_000), rays=_log(rng, 1_000, 4_000_000),
                    variant=rng.choice([0, 1]), block=rng.choice([64, 128, 256]), refill=rng.choice([0, 16, 32]))
    w = _log(rng, 96, 1280)
    h = max(64, int(w * rng.uniform(0.5, 1.0)))
    if kind == "reference":
        return dict(kind=kind, subdiv=rng.randint(2, 6), w=w, h=h, spp=rng.randint(1, 16), depth=rng.randint(4, 12))
    if kind == "viewer":
        return dict(kind=kind, subdiv=rng.randint(2, 6), w=w, h=h, frames=rng.randint(1, 6), depth=rng.randint(6, 12))
    if kind == "path":
        scene = rng.choice(["room", "sky"])
        return dict(kind=kind, scene=scene, subdiv=rng.randint(4, 7) if scene == "sky" else 0, w=w, h=h,
                    spp=rng.randint(1, 32), depth=rng.randint(4, 16))
    if kind == "guided":
        return dict(kind=kind, subdiv=rng.randint(3, 6), w=min(w, 960), h=min(h, 540), spp=rng.randint(4, 24),
                    depth=rng.randint(4, 12), paths=_log(rng, 4_096, 65_536), batch=_log(rng, 8_192, 131_072),
                    bounces=rng.choice([0, 1, 2]))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(2, 8), tri_lo=500, tri_hi=_log(rng, 5_000, 100_000),
                    res=_log(rng, 100, 512), spp=rng.randint(1, 16), depth=rng.randint(4, 10))
    return dict(kind=kind, rows=_log(rng, 100, 1_000_000 if kind == "guide_forward" else 262_144))


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=None)
def _context():
    return tt.Context(0)


@functools.lru_cache(maxsize=None)
def _soup(tris):
    """Equilateral triangles, centroids uniform in the unit cube, log-normal side (0.01 at
    a million triangles, scaled to keep the density), uniform orientation: (tris, 3, 3)."""
    rng = np.random.default_rng([GEO_SEED, tris])
    c = rng.random((tris, 3))
    side = np.exp(rng.normal(math.log(0.01 * (1e6 / tris) ** (1 / 3)), 0.5, tris))
    n = rng.normal(size=(tris, 3))
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    a = np.where(np.abs(n[:, :1]) < 0.9, np.array([[1.0, 0, 0]]), np.array([[0, 1.0, 0]]))
    u = np.cross(n, a)
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    v = np.cross(n, u)
    spin = rng.random(tris) * 2 * math.pi
    pts = [c + (side / math.sqrt(3))[:, None] * (np.cos(spin + k * 2 * math.pi / 3)[:, None] * u +
                                                 np.sin(spin + k * 2 * math.pi / 3)[:, None] * v) for k in range(3)]
    return np.stack(pts, 1).astype(np.float32)


@functools.lru_cache(maxsize=4)
def _soup_tree(tris):
    p = _soup(tris)
    mesh = tt.Mesh.from_arrays(p.reshape(-1, 3), np.arange(3 * tris, dtype=np.int32).reshape(-1, 3))
    return mesh, tt.BVH.build(mesh)


def _surface_points(tris, n, g):
    """n points on random triangles of the soup with their front normals, on the GPU."""
    p = torch.from_numpy(_soup(tris)).to(DEV)
    p = p[torch.randint(tris, (n,), generator=g, device=DEV)]
    r = torch.rand((n, 2), generator=g, device=DEV)
    s = r[:, :1].sqrt()
    at = p[:, 0] * (1 - s) + p[:, 1] * (s * (1 - r[:, 1:])) + p[:, 2] * (s * r[:, 1:])
    nrm = torch.nn.functional.normalize(torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]), dim=1)
    return at, nrm


def _rays(case, seed):
    """Camera rays, then cosine-distributed rays from surface points: float32 (n, 8)."""
    prim = torch.from_numpy(tt.rays_primary(case["w"], case["h"], case["spp"], EYE, (0.5, 0.5, 0.0), fovx=45.0, tmin=0.0,
                                            tmax=16.0, seed=seed)).to(DEV)
    g = torch.Generator(DEV).manual_seed(seed)
    at, nrm = _surface_points(case["tris"], case["scattered"], g)
    d = torch.randn(at.shape, generator=g, device=DEV)
    d = torch.nn.functional.normalize(torch.nn.functional.normalize(d, dim=1) + nrm * 1.0001, dim=1)
    lo = torch.full((len(at), 1), 1e-4, device=DEV)
    hi = torch.full((len(at), 1), 16.0, device=DEV)
    return torch.cat([prim, torch.cat([at, lo, d, hi], 1)]).contiguous()


def _shadow_rays(case, seed):
    """Rays from surface points towards a square light above the scene, ending at it."""
    g = torch.Generator(DEV).manual_seed(seed)
    at, nrm = _surface_points(case["tris"], case["rays"], g)
    at = at + nrm * 1e-4
    light = torch.rand(at.shape, generator=g, device=DEV) * torch.tensor([1.0, 0.0, 1.0], device=DEV)
    light = light + torch.tensor([0.0, 2.0, 0.0], device=DEV)
    d = light - at
    dist = d.norm(dim=1, keepdim=True)
    zero = torch.zeros_like(dist)
    return torch.cat([at, zero, d / dist, dist * (1 - 1e-3)], 1).contiguous()


@functools.lru_cache(maxsize=None)
def _scene_data(scene, subdiv, w, h):
    """(mesh, tree, materials, env, geometries, camera) of a render case."""
    env, geoms = None, []
    if scene == "cornell":
        mesh, mats, cam = workloads.cornell(subdiv=subdiv, width=w, height=h)
    elif scene == "analytic":
        mesh, mats, geoms, cam = workloads.cornell_analytic(width=w, height=h, subdiv=subdiv)
    elif scene == "room":
        mesh, mats, cam = workloads.door_room(width=w, height=h)
    else:
        mesh, mats, env, cam = workloads.pathtrace(subdiv=subdiv, width=w, height=h,
                                                   env_w=2048 if subdiv >= 8 else 512, env_h=1024 if subdiv >= 8 else 256)
    return mesh, tt.BVH.build(mesh), mats, env, geoms, cam


@functools.lru_cache(maxsize=4)
def _batch_data(n, lo, hi, res):
    meshes, mats, cams, env, counts = workloads.batched(n=n, seed=GEO_SEED, tri_lo=lo, tri_hi=hi,
                                                        resolutions=(max(2, res // 2), res))
    return meshes, [tt.BVH.build(m) for m in meshes], mats, cams, env, counts


LAYERS = [(224, 64), (64, 64), (64, 64), (64, 48)]


def _network(seed):
    """Parameters of the guiding network (per layer W[out][in], then b[out])."""
    rng = np.random.default_rng([GEO_SEED, seed])
    out = []
    for k, (i, o) in enumerate(LAYERS):
        w = rng.normal(0.0, (0.3 if k == 3 else 1.0) * math.sqrt(2.0 / i), (o, i))
        b = rng.normal(0.0, 0.05, o)
        if k == 3:
            w[40:], b[40:] = 0.0, 0.0
        out += [w.reshape(-1), b]
    return np.concatenate(out).astype(np.float32)


def _training_rows(rows, seed):
    """Network inputs (position, normal, outgoing direction in [0, 1]), directions and
    radiance weights as a renderer's path records give them."""
    rng = np.random.default_rng([2, seed])

    def unit(n):
        d = rng.normal(size=(n, 3))
        return d / np.linalg.norm(d, axis=1, keepdims=True)
    x = np.concatenate([rng.random((rows, 3)), 0.5 * (unit(rows) + 1), 0.5 * (unit(rows) + 1)], 1)
    return x.astype(np.float32), unit(rows).astype(np.float32), rng.gamma(1.0, 1.0, rows).astype(np.float32)


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    kind, ctx = case["kind"], _context()
    if kind in ("intersect", "closest", "any"):
        mesh, bvh = _soup_tree(case["tris"])
        rays = _shadow_rays(case, seed) if kind == "any" else _rays(case, seed)
        state = dict(case=case, scene=tt.DeviceScene(ctx, mesh, bvh), n=len(rays))
        if kind == "intersect":
            state["rays"] = rays.cpu().numpy()
            state["cfg"] = None if case["variant"] == 0 else tt.trace_cfg(1)
            return state
        state["rays"] = rays
        state["out"] = torch.zeros((len(rays), 4) if kind == "closest" else (len(rays),),
                                   dtype=torch.float32 if kind == "closest" else torch.int32, device=DEV)
        default = (case["variant"], case["block"], case["refill"], case.get("reorder", 0)) == (0, 128, 0, 0)
        state["cfg"] = None if default else tt.trace_cfg(case["variant"], 16, case["block"], refill=case["refill"],
                                                         reorder=case.get("reorder", 0))
        torch.cuda.synchronize()
        return state
    if kind in ("reference", "viewer", "path", "guided"):
        name = {"reference": "cornell", "viewer": "analytic", "guided": "sky"}.get(kind) or case["scene"]
        mesh, bvh, mats, env, geoms, cam = _scene_data(name, case["subdiv"], case["w"], case["h"])
        scene = tt.DeviceScene(ctx, mesh, bvh, mats, env=env)
        if geoms:
            scene.set_geometries(geoms)
        state = dict(case=case, scene=scene, cam=cam, seed=seed)
        if kind == "viewer":
            state["display"] = tt.Display(ctx, case["w"], case["h"])
        elif kind == "reference":
            state["params"] = tt.render_params(spp=case["spp"], max_depth=case["depth"], seed=seed,
                                               mode=tt.RENDER_REFERENCE)
        else:
            state["params"] = tt.render_params(spp=case["spp"], max_depth=case["depth"], rr_depth=4, seed=seed,
                                               mode=tt.RENDER_PATH,
                                               paths_in_flight=case["w"] * case["h"] if kind == "guided" else 0)
        if kind == "guided":
            state["guide"] = tt.Guide(ctx, seed=seed, lr=1e-3)
        return state
    if kind == "batch":
        meshes, bvhs, mats, cams, env, _ = _batch_data(case["scenes"], case["tri_lo"], case["tri_hi"], case["res"])
        return dict(case=case, batch=tt.Batch(ctx, meshes, bvhs, mats, env=env), cams=cams,
                    params=tt.render_params(spp=case["spp"], max_depth=case["depth"], rr_depth=4, seed=seed,
                                            mode=tt.RENDER_PATH))
    guide = tt.Guide(ctx, seed=3, lr=1e-3)
    guide.set_params(_network(seed))
    return dict(case=case, guide=guide, rows=_training_rows(case["rows"], seed))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "intersect":
        ids, t, u, v = state["scene"].intersect(state["rays"], state["cfg"])
        return dict(id=ids, t=t, u=u, v=v)
    if kind == "closest":
        out = state["out"]
        state["scene"].trace_closest(state["rays"].data_ptr(), state["n"], out.data_ptr(), state["cfg"])
        return dict(id=out.view(torch.int32)[:, 0], t=out[:, 1], u=out[:, 2], v=out[:, 3])
    if kind == "any":
        state["scene"].trace_any(state["rays"].data_ptr(), state["n"], state["out"].data_ptr(), state["cfg"])
        return dict(hit=state["out"])
    if kind == "viewer":
        display = state["display"]
        display.reset()
        for k in range(case["frames"]):
            params = tt.render_params(spp=1, max_depth=case["depth"], seed=state["seed"] + k, mode=tt.RENDER_REFERENCE)
            img, _ = state["scene"].render(state["cam"], params)
            rgba = display.frame(img)
        return dict(frame=img, rgba=rgba)
    if kind in ("reference", "path"):
        img, _ = state["scene"].render(state["cam"], state["params"])
        return dict(image=img)
    if kind == "guided":
        guide = state["guide"]
        img, _, _ = guide.render(state["scene"], state["cam"], state["params"], train=True, train_paths=case["paths"],
                                 train_batch=case["batch"], max_bounce=case["bounces"], pass_growth=8, learn_alpha=True)
        return dict(image=img, params=guide.params())
    if kind == "batch":
        imgs, _ = state["batch"].render(state["cams"], state["params"])
        return dict(images=imgs)
    guide, (x, d, w) = state["guide"], state["rows"]
    if kind == "guide_forward":
        return dict(raw=guide.forward(x))
    loss = guide.train_step(x, d, w)
    return dict(loss=loss, params=guide.params())


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind = case["kind"]
    # a traversal cannot do with less than a walk down one path of the tree, two boxes a
    # level, and a few triangle tests; about 20 and 40 operations each
    def per_ray(tris):
        return 40.0 * math.log2(max(2, tris)) + 160.0
    if kind in ("intersect", "closest"):
        n = case["w"] * case["h"] * case["spp"] + case["scattered"]
        return dict(bytes=48.0 * n + 36.0 * case["tris"], flops=n * per_ray(case["tris"]))
    if kind == "any":
        return dict(bytes=36.0 * case["rays"] + 36.0 * case["tris"], flops=case["rays"] * per_ray(case["tris"]))
    macs = sum(i * o for i, o in LAYERS)
    params = sum(i * o + o for i, o in LAYERS)
    if kind in ("reference", "viewer", "path", "guided"):
        sky = kind == "guided" or (kind == "path" and case["scene"] == "sky")
        tris = 20 * 4 ** case["subdiv"] if (kind != "path" or sky) else 20
        samples = case["w"] * case["h"] * (case["frames"] if kind == "viewer" else case["spp"])
        # open scene: about 2.5 rays a sample (sky hits end paths); closed: most of the depth
        rays = samples * (2.5 if sky else 0.7 * case["depth"])
        pixels = case["w"] * case["h"] * (28.0 * case["frames"] if kind == "viewer" else 12.0)
        # guided: about a third of the vertices of the guided bounces go through the network
        net = samples * 2.0 * macs / 3 if kind == "guided" else 0.0
        return dict(bytes=pixels + 68.0 * tris, flops=rays * (per_ray(tris) + 300.0) + net)
    if kind == "batch":
        _, _, _, cams, _, counts = _batch_data(case["scenes"], case["tri_lo"], case["tri_hi"], case["res"])
        pixels = sum(c.width * c.height for c in cams)
        return dict(bytes=12.0 * pixels + 68.0 * sum(counts),
                    flops=sum(2.5 * c.width * c.height * case["spp"] * (per_ray(k) + 300.0) for c, k in zip(cams, counts)))
    if kind == "guide_forward":
        return dict(bytes=case["rows"] * (36.0 + 160.0) + 4.0 * params, flops=2.0 * macs * case["rows"])
    return dict(bytes=case["rows"] * 52.0 + 28.0 * params, flops=6.0 * macs * case["rows"])


# ------------------------------------------------------------------ the same in 64 bits
def _exact_closest(case, seed):
    rays = _rays(case, seed).double()
    p = torch.from_numpy(_soup(case["tris"])).to(DEV)
    v0 = p[:, 0].double()
    e1, e2 = (p[:, 1] - p[:, 0]).double(), (p[:, 2] - p[:, 0]).double()
    out = torch.zeros((len(rays), 3), dtype=torch.float64, device=DEV)
    step = max(1, 40_000_000 // case["tris"])
    for at in range(0, len(rays), step):
        r = rays[at:at + step]
        o, lo, d, hi = r[:, None, :3], r[:, 3:4], r[:, None, 4:7], r[:, 7:8]
        pv = torch.linalg.cross(d.expand(-1, len(p), -1), e2[None].expand(len(r), -1, -1))
        det = (e1[None] * pv).sum(2)
        tv = o - v0[None]
        u = (tv * pv).sum(2) / det
        del pv
        qv = torch.linalg.cross(tv, e1[None].expand(len(r), -1, -1))
        v = (d * qv).sum(2) / det
        t = (e2[None] * qv).sum(2) / det
        ok = (det > 1e-5) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1) & (t > lo) & (t < hi)
        t, k = torch.where(ok, t, math.inf).min(1, keepdim=True)
        hit = torch.isfinite(t)
        out[at:at + step] = torch.cat([torch.where(hit, t, hi), torch.where(hit, u.gather(1, k), 0.0),
                                       torch.where(hit, v.gather(1, k), 0.0)], 1)
    return out


def _exact_network(params, x):
    """The 40 outputs for inputs x in 64 bits."""
    f = torch.arange(12, device=x.device, dtype=torch.float64)
    a = math.pi * x[:, :, None] * 2.0 ** f
    h = torch.stack([a.sin(), a.cos()], 3).reshape(len(x), 216)
    at = 0
    for k, (i, o) in enumerate(LAYERS):
        w = params[at:at + i * o].reshape(o, i)
        b = params[at + i * o:at + i * o + o]
        at += i * o + o
        h = h @ w[:, :h.shape[1]].T + b
        if k < 3:
            h = h.clamp(min=0)
    return h[:, :40]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("intersect", "closest"):
        n = case["w"] * case["h"] * case["spp"] + case["scattered"]
        if n * case["tris"] > 2_000_000_000:
            return None
        out = _exact_closest(case, seed)
        return dict(id=None, t=out[:, 0], u=out[:, 1], v=out[:, 2])
    if kind == "guide_forward":
        x, _, _ = _training_rows(case["rows"], seed)
        p = torch.from_numpy(_network(seed)).to(DEV).double()
        x = torch.from_numpy(x).to(DEV).double()
        return dict(raw=torch.cat([_exact_network(p, part) for part in x.split(65536)]))
    if kind == "guide_train":
        x, d, w = (torch.from_numpy(a).to(DEV).double() for a in _training_rows(case["rows"], seed))
        p = torch.from_numpy(_network(seed)).to(DEV).double()
        total, norm = 0.0, w.sum()
        for px, pd, pw in zip(x.split(65536), d.split(65536), w.split(65536)):
            raw = _exact_network(p, px)
            m = raw[:, :24].reshape(-1, 8, 3)
            mu = m / (m.norm(dim=2, keepdim=True) + 1e-6)
            kappa = raw[:, 24:32].clamp(-5.0, 9.0).exp()
            c = (mu * pd[:, None]).sum(2)
            lv = (raw[:, 32:40].log_softmax(1) + kappa.log() - math.log(2 * math.pi) -
                  torch.log1p(-torch.exp(-2 * kappa)) + kappa * (c - 1))
            total = total - (pw * torch.logsumexp(lv, 1)).sum() / norm
        return dict(loss=total, params=None)
    return None
